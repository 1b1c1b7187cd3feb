// Convolution: tensor_conv (src/convolution.cpp:34-100) and vulkan_conv
// (src/backend_vulkan.cpp:1177-1209, :1359-1402) as an implicit GEMM on bf16
// MFMA (gfx950).
//
// The reference forms the im2col patches of every output pixel (inner index
// (c * kernel_y + ky) * kernel_x + kx, zero outside the image), multiplies them
// by the float weight [out][inner] in fp32 (cpu_gemm's FMA tiles, or the
// Vulkan matmul shader) and adds the bias.  Here the patches are never written
// out: a workgroup gathers its 128 pixels x 32 inner values straight from the
// image into LDS, with the inner dimension ordered (ky, kx, c) so that a stage
// of 32 is one kernel tap over 32 consecutive channels (one 128-byte run per
// pixel) whenever channels % 32 == 0 -- the weight is stored in that order
// when it is made resident.  fp32 operands are split into bf16 halves (hi =
// bf16(x), lo = bf16(x - hi)) and a*b = hi*hi + hi*lo + lo*hi on
// v_mfma_f32_32x32x16_bf16 with fp32 accumulation, about 2^-16 relative per
// product.  The matrix core bounds the large layers, so weights that have fewer
// bits than an fp32 take fewer products: BF16 weights are one bf16 plane (two
// products, the same sums), F16 weights one fp16 plane that multiplies an image
// split in fp16 under a scale (two products; conv_body_ring).  256^2 pixels,
// 512 -> 512, 3x3: three products 881 us, two fp16 708 (error against 64 bits
// 4.5e-6 / 6.2e-7), two bf16 665.
//
// Tile: 128 pixels x 128 output channels x 32 inner per stage, 4 waves of
// 64 x 64 (2 x 2 MFMA tiles).  The image kernel (images below 2 GiB) keeps one
// LDS stage of the split image (hi / lo planes, 80-byte rows) and a two-slot
// ring of the weight planes filled by L2 -> LDS transfers, with the image
// loads two stages ahead in registers; it is built for three waves per SIMD
// (at most 168 registers), so three workgroups share a CU.  Larger images and
// channel counts that are not a multiple of 32 take a simpler single-stage
// form (conv_body).

#include <algorithm>

#include "pixhip_device.h"
#include "pixhip_internal.h"


namespace pixhip {

namespace {

typedef __bf16 cbf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t cu32x4 __attribute__((ext_vector_type(4)));

constexpr int kCN = 128, kCK = 32;   // workgroup output channels, inner values per stage
constexpr int kCRow = 40;            // LDS row: 32 bf16 + 8 padding (80 B)

__device__ __forceinline__ uint32_t rne16(float x)
{
    const uint32_t u = __float_as_uint(x);
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

// x -> (hi, lo) bf16 with x ~ hi + lo for every fp32 value (the weight form
// and the value-by-value gather): a finite x that rounds past the largest
// bf16 keeps hi truncated; Inf and NaN travel in hi alone (lo = 0).  The image
// kernel's hardware split (halves2) assumes finite values that round to a
// finite bf16, |x| < (2 - 2^-8) * 2^127 ~ 3.396e38: beyond that, and for Inf
// and NaN, its halves give NaN.
__device__ __forceinline__ void halves(float x, uint32_t& hi, uint32_t& lo)
{
    const uint32_t u = __float_as_uint(x);
    if ((u & 0x7F800000u) == 0x7F800000u) {
        hi = (u & 0x007FFFFFu)? 0x7FC0u | ((u >> 16) & 0x8000u) : u >> 16;
        lo = 0;
        return;
    }
    uint32_t h = rne16(x);
    if ((h & 0x7F80u) == 0x7F80u) h = u >> 16;
    hi = h;
    lo = rne16(x - __uint_as_float(h << 16));
}

typedef __bf16 cbf16x2 __attribute__((ext_vector_type(2)));
typedef __amdgpu_buffer_rsrc_t CRsrc;

// One 1 KB L2 -> LDS transfer (lane l's 16 bytes to lds_dst + 16 l), written
// as asm: issued through the builtin, the compiler makes every later LDS
// access wait for all transfers in flight (it cannot tell them apart), which
// would undo the ring.  The waits for these transfers are the explicit ones
// before the barriers; the compiler's own counts for the image loads only
// grow stronger from operations it does not see (the counter is in order).
// s_nop 0: one wait state between writing M0 and the transfer that reads it.
__device__ __forceinline__ void conv_dma(CRsrc r, const uint16_t* lds_dst, uint32_t voff, uint32_t soff)
{
    const uint32_t m = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint16_t*)lds_dst;
    __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :: "s"(__builtin_amdgcn_readfirstlane(m)), "v"(voff), "s"(r), "s"(__builtin_amdgcn_readfirstlane(soff))
                     : "memory", "m0");
}

// s_waitcnt vmcnt(N) lgkmcnt(0), then s_barrier: the wave's own LDS reads
// and writes are done and all but its N newest vector-memory operations
// (loads and L2 -> LDS transfers, counted in issue order) have completed.
// (__syncthreads' workgroup fence must complete the wave's LDS writes, and
// with the compiler's L2 -> LDS transfers in flight that means every
// outstanding vector-memory operation.)
template <int N> __device__ __forceinline__ void conv_barrier()
{
    static_assert(N >= 0 && N < 16, "vmcnt range");
    __builtin_amdgcn_s_waitcnt(N | (7 << 4) | (0 << 8));
    __builtin_amdgcn_s_barrier();
}

// Raw buffer of `bytes` bytes (stride 0): loads at or past the end read zeros.
__device__ __forceinline__ CRsrc conv_rsrc(const void* base, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base),(short)0,(int)bytes,0x00020000);
}

// Two values rounded to bf16 (nearest even) by v_cvt_pk_bf16_f32; a in the
// low half.  For finite values the same bits as rne16.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b)
{
    const cbf16x2 h = {(__bf16)a,(__bf16)b};
    return __builtin_bit_cast(uint32_t,h);
}

// The split of a pair: hi = both values rounded to bf16, lo = the remainders
// rounded to bf16 (six vector instructions for two values).
__device__ __forceinline__ void halves2(float a, float b, uint32_t& hi, uint32_t& lo)
{
    hi = pack_bf16(a,b);
    lo = pack_bf16(a - __uint_as_float(hi << 16),b - __uint_as_float(hi & 0xFFFF0000u));
}

// Eight fp16 values as bf16 halves (exact: 11 bits are 8 and 3).
__device__ __forceinline__ void half_planes(cu32x4 v, cu32x4& hi, cu32x4& lo)
{
    const v8h h = __builtin_bit_cast(v8h,v);
    uint32_t a[4], b[4];
#pragma unroll
    for (int q = 0; q < 4; q++) halves2((float)h[2 * q],(float)h[2 * q + 1],a[q],b[q]);
    hi = cu32x4{a[0],a[1],a[2],a[3]};
    lo = cu32x4{b[0],b[1],b[2],b[3]};
}

// The fp16 split of a pair times `scale` (a power of two): hi truncated to fp16,
// lo = the remainders truncated to fp16: 2^-20 of the value, or fp16's last place
// 2^-24 where that is more.  (The remainders as fused multiply-adds of the
// unscaled values: the same exact differences, one mixed-precision instruction
// each.)
__device__ __forceinline__ void halves2_f16(float a, float b, float scale, uint32_t& hi, uint32_t& lo)
{
    const auto h = __builtin_amdgcn_cvt_pkrtz(a * scale,b * scale);
    hi = __builtin_bit_cast(uint32_t,h);
    lo = __builtin_bit_cast(uint32_t,__builtin_amdgcn_cvt_pkrtz(__builtin_fmaf(a,scale,-(float)h[0]),__builtin_fmaf(b,scale,-(float)h[1])));
}

__device__ __forceinline__ float weight_value(const uint8_t* raw, uint32_t type, size_t index)
{
    if (type == PIX_F32) {
        const uint8_t* p = raw + 4 * index;
        return __uint_as_float((uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24));
    }
    const uint8_t* p = raw + 2 * index;
    const uint16_t h = (uint16_t)(p[0] | (p[1] << 8));
    return type == PIX_F16? half_bits_to_float(h) : __uint_as_float((uint32_t)h << 16);
}

}  // namespace

// The form a weight of `type` is held in: BF16 weights are one bf16 plane, F16
// weights one fp16 plane where the image kernel reads them (whole stages of 32
// channels), everything else the two split planes.
int conv_weight_kind(uint32_t type, int cin)
{
    if (type == PIX_BF16) return kConvBf16;
    return type == PIX_F16 && cin % kCK == 0? kConvHalf : kConvSplit;
}

// Weight form: planes [npad][kp] of bf16 (hi, lo; the fp16 or bf16 plane alone
// where the weight has only one); row n, column k' = (ky *
// kernel_x + kx) * cin + c holds weight[n][(c * kernel_y + ky) * kernel_x + kx]
// of the GGUF / safetensors tensor; zero past cout and inner.
__global__ __launch_bounds__(256) void conv_form_kernel(const uint8_t* __restrict__ raw, uint32_t type, int kx_n, int ky_n, int cin,
                                                        int cout, int kp, int npad, int kind, uint16_t* __restrict__ hi, uint16_t* __restrict__ lo)
{
    const size_t inner = (size_t)cin * kx_n * ky_n, total = (size_t)npad * kp, step = (size_t)gridDim.x * blockDim.x;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += step) {
        const int n = (int)(e / kp), k = (int)(e % kp);
        float w = 0.0f;
        if (n < cout && (size_t)k < inner) {
            const int c = k % cin, tap = k / cin, kx = tap % kx_n, ky = tap / kx_n;
            w = weight_value(raw,type,(size_t)n * inner + ((size_t)c * ky_n + ky) * kx_n + kx);
        }
        if (kind == kConvHalf) {
            hi[e] = float_to_half_bits(w);  // (exact: the value was fp16)
            continue;
        }
        uint32_t h, l;
        halves(w,h,l);
        hi[e] = (uint16_t)h;
        if (kind == kConvSplit) lo[e] = (uint16_t)l;
    }
}

// sums[n] = sum of |w| over row n of an fp16 plane, one wave per row.
__global__ __launch_bounds__(64) void conv_row_sums_kernel(const uint16_t* __restrict__ plane, int kp, float* __restrict__ sums)
{
    float v = 0.0f;
    for (int k = 8 * (int)threadIdx.x; k < kp; k += 512) {
        const v8h h = *reinterpret_cast<const v8h*>(plane + (size_t)blockIdx.x * kp + k);
#pragma unroll
        for (int i = 0; i < 8; i++) v += __builtin_fabsf((float)h[i]);
    }
    v = wave_sum(v);
    if (threadIdx.x == 0) sums[blockIdx.x] = v;
}

hipError_t launch_conv_form(const void* raw, uint32_t type, int kernel_x, int kernel_y, int cin, int cout, int kp, int npad, int kind,
                            uint16_t* hi, uint16_t* lo, float* sums, hipStream_t s)
{
    const size_t total = (size_t)npad * kp;
    const unsigned grid = (unsigned)std::min<size_t>((total + 255) / 256,(size_t)1 << 20);
    conv_form_kernel<<<dim3(grid),dim3(256),0,s>>>(static_cast<const uint8_t*>(raw),type,kernel_x,kernel_y,cin,cout,kp,npad,kind,hi,lo);
    if (kind == kConvHalf) conv_row_sums_kernel<<<dim3((unsigned)npad),dim3(64),0,s>>>(hi,kp,sums);
    return hipGetLastError();
}

// MODE 1: cin % 32 == 0 and the image 16-byte aligned (a stage is one tap of
// 32 consecutive channels, read as float4) at 64-bit addresses, for images of
// 2 GiB and more; MODE 0: each inner value is gathered on its own (the first
// layer's 3 or 16 channels).  The next stage's loads are held in registers
// while the current one is multiplied.  Each wave owns MT = 2 tiles of 32
// pixels by 2 of 32 channels (a 256-pixel workgroup tile with 128 x 64 per
// wave ran 27% slower).
template <int MODE>
__device__ __forceinline__ void conv_body(const ConvArgs& a)
{
    constexpr bool FAST = MODE != 0;
    constexpr int MT = 2;
    constexpr int BM = 64 * MT;                        // workgroup pixels
    constexpr int PA = BM * kCRow, PB = kCN * kCRow;   // bf16 per A / B plane
    constexpr int STAGE = 2 * PA + 2 * PB;
    constexpr int AV = FAST? BM * 8 / 256 : BM * 32 / 256;  // A values (float4 or scalar) per thread
    __shared__ __attribute__((aligned(16))) uint16_t lds[STAGE];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, lr = lane & 31, hh = lane >> 5;
    const int wm = wave & 1, wn = wave >> 1;
    const long long m0 = (long long)blockIdx.x * BM;
    const int n0 = blockIdx.y * kCN;

    // the pixels this thread loads: rows t/8 + 32i (FAST), rows t/32 + 8i (gather)
    int iy0[AV], ix0[AV];
#pragma unroll
    for (int i = 0; i < AV; i++) {
        const long long m = m0 + (FAST? t / 8 + 32 * i : t / 32 + 8 * i);
        if (m < a.M) {
            const int oy = (int)(m / a.OW), ox = (int)(m % a.OW);
            iy0[i] = oy * a.SY - a.PT;
            ix0[i] = ox * a.SX - a.PL;
        } else {
            iy0[i] = -(1 << 30);  // never inside the image
            ix0[i] = 0;
        }
    }

    float4 ra[FAST? AV : 1];
    bool ain[FAST? AV : 1];
    float rs[FAST? 1 : AV];
    cu32x4 rb[4];
    auto fetch = [&](int stage) {
        const int k0 = stage * kCK;
        if constexpr (FAST) {
            const int tap = k0 / a.C, c = k0 % a.C + (t % 8) * 4;
            const int ky = tap / a.KX, kx = tap % a.KX;
            // every lane loads: a tap outside the image reads pixel 0 and
            // store() puts zeros in its place, so no load sits behind a branch
#pragma unroll
            for (int i = 0; i < AV; i++) {
                const int iy = iy0[i] + ky, ix = ix0[i] + kx;
                ain[i] = iy >= 0 && iy < a.H && ix >= 0 && ix < a.W;
                const unsigned pix = ain[i]? (unsigned)iy * (unsigned)a.W + (unsigned)ix : 0u;  // < 2^32 pixels
                ra[i] = *reinterpret_cast<const float4*>(a.x + (size_t)pix * a.C + c);
            }
        } else {
            const int k = k0 + t % 32;
            const int c = k % a.C, tap = k / a.C, ky = tap / a.KX, kx = tap % a.KX;
#pragma unroll
            for (int i = 0; i < AV; i++) {
                const int iy = iy0[i] + ky, ix = ix0[i] + kx;
                rs[i] = (k < a.K && iy >= 0 && iy < a.H && ix >= 0 && ix < a.W) ? a.x[((size_t)iy * a.W + ix) * a.C + c] : 0.0f;
            }
        }
        // B: 128 rows x 64 bytes per plane, two 16-byte pieces per thread per plane
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int q = t + 256 * (j & 1), row = q / 4, part = q % 4;
            if (j >= 2 && a.kind != kConvSplit) continue;  // one plane
            const uint16_t* plane = (j < 2)? a.wh : a.wl;
            rb[j] = *reinterpret_cast<const cu32x4*>(plane + (size_t)(n0 + row) * a.Kp + k0 + part * 8);
        }
    };
    auto store = [&]() {
        uint16_t* st = lds;
        if constexpr (FAST) {
#pragma unroll
            for (int i = 0; i < AV; i++) {
                const int row = t / 8 + 32 * i, col = (t % 8) * 4;
                const float4 v = ain[i]? ra[i] : make_float4(0.0f,0.0f,0.0f,0.0f);
                uint32_t h01, l01, h23, l23;
                halves2(v.x,v.y,h01,l01);
                halves2(v.z,v.w,h23,l23);
                *reinterpret_cast<uint2*>(st + row * kCRow + col) = make_uint2(h01,h23);
                *reinterpret_cast<uint2*>(st + PA + row * kCRow + col) = make_uint2(l01,l23);
            }
        } else {
#pragma unroll
            for (int i = 0; i < AV; i++) {
                const int row = t / 32 + 8 * i, col = t % 32;
                uint32_t h, l;
                halves(rs[i],h,l);
                st[row * kCRow + col] = (uint16_t)h;
                st[PA + row * kCRow + col] = (uint16_t)l;
            }
        }
        if (a.kind == kConvHalf) {
#pragma unroll
            for (int j = 0; j < 2; j++) half_planes(rb[j],rb[j],rb[j + 2]);
        } else if (a.kind == kConvBf16) {
            rb[2] = rb[3] = cu32x4{0,0,0,0};
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int q = t + 256 * (j & 1), row = q / 4, part = q % 4;
            *reinterpret_cast<cu32x4*>(st + 2 * PA + (j >> 1) * PB + row * kCRow + part * 8) = rb[j];
        }
    };

    v16f acc[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = v16f{};

    const int stages = a.Kp / kCK;
    fetch(0);
    store();
    __syncthreads();
    for (int s = 0; s < stages; s++) {
        if (s + 1 < stages) fetch(s + 1);
        const uint16_t* st = lds;
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            const int col = ks * 16 + 8 * hh;
            cbf16x8 ah[MT], al[MT], bh[2], bl[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int row = wn * 64 + j * 32 + lr;
                bh[j] = *reinterpret_cast<const cbf16x8*>(st + 2 * PA + row * kCRow + col);
                bl[j] = *reinterpret_cast<const cbf16x8*>(st + 2 * PA + PB + row * kCRow + col);
            }
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const int row = wm * (BM / 2) + i * 32 + lr;
                ah[i] = *reinterpret_cast<const cbf16x8*>(st + row * kCRow + col);
                al[i] = *reinterpret_cast<const cbf16x8*>(st + PA + row * kCRow + col);
            }
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i],bh[j],acc[i][j],0,0,0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i],bl[j],acc[i][j],0,0,0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[i],bh[j],acc[i][j],0,0,0);
                }
        }
        if (s + 1 < stages) {
            __syncthreads();  // every wave is done reading the stage
            store();
            __syncthreads();
        }
    }

    // acc[i][j] lane: output channel n0 + wn*64 + 32j + lr, pixels
    // m0 + wm*BM/2 + 32i + 8(r/4) + 4hh + r%4
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int n = n0 + wn * 64 + 32 * j + lr;
        if (n >= a.N) continue;
        const float b = a.bias? a.bias[n] : 0.0f;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const long long m = m0 + wm * (BM / 2) + 32 * i + 8 * (r / 4) + 4 * hh + r % 4;
                if (m < a.M) a.y[(size_t)m * a.N + n] = a.bias? __fadd_rn(acc[i][j][r],b) : acc[i][j][r];
            }
    }
}


// How a tile of the fp16 form is held, from a sample of its inner range: the
// centre tap's first 32 channels and, where an output is not held by those, the
// first 32 of the other taps in turn.
//   scale  a power of two from the largest |x| at the centre tap, in steps of
//          2^2: 2^7 for 2 .. 8, so that neighbouring tiles, and the same values
//          at another place of another image, mostly split alike.  The largest
//          becomes 2^8 .. 2^10: 64 times as much still fits fp16, and a pixel of
//          normal values may be 50 times dimmer than the tile's brightest (at
//          4608 inner values) before it is not held.  0 where an output whose
//          pixel is not blank is not held: its share of the sum |x| |w| in the
//          sample is less than kLeast of its sum |w|;
//   blank  bit i: the sample holds only zeros for this thread's pixel t / 8 + 32 i.
// With FURTHER false only the centre tap is looked at, and scale is 0 unless it
// holds every output (all but a few tiles): a stage without its pipelining, and
// half of its products.
constexpr float kLeast = 1.01f / 128;  // 2^-7, and 1% for the sum's rounding
struct ConvProbe {
    float scale;
    int blank;
};
template <bool FURTHER>
__device__ __forceinline__ ConvProbe conv_probe(const ConvArgs& a, uint16_t* lds, uint16_t* bs)
{
    // (opaque: values shared with the loop would sit in registers through it)
    int t = threadIdx.x;
    uint32_t tile_m = blockIdx.x, tile_n = blockIdx.y;
    __asm__ volatile("" : "+v"(t), "+s"(tile_m), "+s"(tile_n));
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), lr = lane & 31, hh = lane >> 5;
    const int wm = wave & 1, wn = wave >> 1;
    const long long m0 = (long long)tile_m * 128;
    const int n0 = (int)tile_n * kCN, taps = FURTHER? a.KX * a.KY : 1, centre = a.KY / 2 * a.KX + a.KX / 2;
    float* const waves = reinterpret_cast<float*>(lds + 128 * kCRow);  // [4]
    float* const most = waves + 4;                                     // [128]: the pixels' maxima (FURTHER)
    ConvProbe probe = {0.0f,0};
    float row[4] = {0.0f,0.0f,0.0f,0.0f};
    v16f sum[2][2] = {};
    bool held = true, lost = false;
    for (int p = 0; p < taps; p++) {
        const int tap = p == 0? centre : p <= centre? p - 1 : p;
        const int ky = tap / a.KX, kx = tap % a.KX;
        cu32x4 rb[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int q = t + 256 * j;
            rb[j] = *reinterpret_cast<const cu32x4*>(a.wh + (size_t)(n0 + q / 4) * a.Kp + (size_t)tap * a.C + 8 * (q % 4));
        }
        float4 ra[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t m = (uint32_t)m0 + t / 8 + 32 * i, oy = m / (uint32_t)a.OW, ox = m - oy * (uint32_t)a.OW;
            const int iy = (int)oy * a.SY - a.PT + ky, ix = (int)ox * a.SX - a.PL + kx;
            ra[i] = make_float4(0.0f,0.0f,0.0f,0.0f);
            if (m < a.M && iy >= 0 && iy < a.H && ix >= 0 && ix < a.W)
                ra[i] = *reinterpret_cast<const float4*>(a.x + ((size_t)iy * a.W + ix) * a.C + (t % 8) * 4);
            float v = __builtin_fmaxf(__builtin_fabsf(ra[i].x),__builtin_fabsf(ra[i].y));
            v = __builtin_fmaxf(__builtin_fmaxf(v,__builtin_fabsf(ra[i].z)),__builtin_fabsf(ra[i].w));
            v = __builtin_fmaxf(v,dpp_f32<kDppXor1>(v));
            v = __builtin_fmaxf(v,dpp_f32<kDppXor2>(v));
            row[i] = __builtin_fmaxf(row[i],__builtin_fmaxf(v,dpp_f32<kDppHalfMirror>(v)));
        }
        if (p == 0) {
            float v = __builtin_fmaxf(__builtin_fmaxf(row[0],row[1]),__builtin_fmaxf(row[2],row[3]));
            v = __builtin_fmaxf(v,dpp_f32<kDppMirror>(v));
            v = __builtin_fmaxf(__builtin_fmaxf(lane_f32(v,0),lane_f32(v,16)),__builtin_fmaxf(lane_f32(v,32),lane_f32(v,48)));
            if (lane == 0) waves[wave] = v;
            __syncthreads();
            v = __builtin_fmaxf(__builtin_fmaxf(waves[0],waves[1]),__builtin_fmaxf(waves[2],waves[3]));
            const int e = (int)(__float_as_uint(v) >> 23);  // biased exponent: 2^(e - 127) <= v
            const int s = e == 0 || e == 255? 134 : min(134 - ((e - 128) >> 1) * 2,250);  // (8 .. 250: a normal power of two)
            probe.scale = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane(s) << 23);
        }
        // |x| * scale (its fp16 hi, not above it) and |w| into LDS, as the ring
        // has them; rows past the image hold fp16's largest
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = t / 8 + 32 * i;
            const bool past = m0 + r >= a.M;
            uint32_t h01, h23, l;
            halves2_f16(__builtin_fabsf(ra[i].x),__builtin_fabsf(ra[i].y),probe.scale,h01,l);
            halves2_f16(__builtin_fabsf(ra[i].z),__builtin_fabsf(ra[i].w),probe.scale,h23,l);
            *reinterpret_cast<uint2*>(lds + r * kCRow + (t % 8) * 4) = past? make_uint2(0x7BFF7BFFu,0x7BFF7BFFu) : make_uint2(h01,h23);
            if (FURTHER && t % 8 == 0) most[r] = past? -1.0f : row[i];
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int q = t + 256 * j, r = q / 4;
            *reinterpret_cast<cu32x4*>(bs + r * 32 + (((q % 4) ^ ((r >> 2) & 3)) << 3)) = rb[j] & 0x7FFF7FFFu;
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            v8h x[2], w[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int r = wn * 64 + j * 32 + lr;
                x[j] = *reinterpret_cast<const v8h*>(lds + (wm * 64 + j * 32 + lr) * kCRow + ks * 16 + 8 * hh);
                w[j] = *reinterpret_cast<const v8h*>(bs + r * 32 + (((2 * ks + hh) ^ ((r >> 2) & 3)) << 3));
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[i],w[j],sum[i][j],0,0,0);
        }
        held = true;
        float far = 0.0f;  // the largest |x| of a pixel with an output that is not held
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float least = a.wsum[n0 + wn * 64 + 32 * j + lr] * kLeast;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                if constexpr (FURTHER) {
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const float m = most[wm * 64 + 32 * i + 8 * (r / 4) + 4 * hh + r % 4];
                        const bool in = (sum[i][j][r] >= least) | (m < 0.0f);
                        held = held & in;
                        far = __builtin_fmaxf(far,in? 0.0f : m);
                    }
                } else {
                    float v = sum[i][j][0];
#pragma unroll
                    for (int r = 1; r < 16; r++) v = __builtin_fminf(v,sum[i][j][r]);
                    held = held & (v >= least);
                }
            }
        }
        lost = far != 0.0f;
        held = __syncthreads_and(held);
        if (held) break;
    }
    if constexpr (FURTHER) {
#pragma unroll
        for (int i = 0; i < 4; i++) probe.blank |= row[i] == 0.0f? 1 << i : 0;
        if (__syncthreads_or(lost)) probe.scale = 0.0f;
    } else if (!held) {
        probe.scale = 0.0f;
    }
    return probe;
}

// The image kernel for images below 2 GiB, pipelined deeper than conv_body:
// the weight planes go L2 -> LDS by buffer_load ... lds into a two-slot ring
// (64-byte rows, piece c of row r at c ^ ((r >> 2) & 3), no registers), and
// the image loads run two stages ahead in two register sets, so a stage's
// stores to LDS wait on loads issued a whole stage earlier.  LDS: one A stage
// (hi, lo: 20 KB) + two B slots (16 KB for hi and lo; the second 8 KB where the
// weight is one plane) = 44 or 52 KB, three workgroups per CU.
//
// FORM is how the products are formed:
//   kConvSplit  three bf16 products of split weights and image;
//   kConvBf16   the weight is one bf16 plane: two products, the same sums;
//   kConvHalf   the weight is one fp16 plane: two fp16 products of the image
//               times `scale` (a power of two), split as hi + lo in fp16, for
//               tiles that can be held this way (conv_probe);
//   kConvWiden  the others: the plane widened to bf16 halves, three bf16
//               products, one stage at a time.
//
// The fp16 split leaves an output an error of at most 2^-20 of its sum |x| |w|
// plus 2^-24 / scale (fp16's last place) of its sum |w|.  The second term must
// stay below 2^-17 of the sum |x| |w| (three bf16 products leave up to 2^-15),
// whatever the magnitudes of the channels and weights are: the sum of the scaled
// image must be kLeast of the sum |w| or more, which conv_probe shows with a
// sample's share of it.  Where a pixel that the sample holds only zeros of has
// other values, or a scaled value leaves fp16's range, kConvHalf returns true,
// without an output.  256^2 pixels, 512 -> 512, 3x3, us: 708 (700 without the
// bound, three products 881); with half of the pixels 2^12 times dimmer, every
// tile on its second try, 954; a border of zeros, whose tiles take the longer
// look, 788 (64^2 pixels: 70, three products 75, with the border 105).
constexpr int kConvWiden = 3;
template <int FORM, int B0, int B1>
__device__ __forceinline__ bool conv_body_ring(const ConvArgs& a, const ConvProbe& probe, uint16_t (&lds)[2 * 128 * kCRow],
                                               uint16_t (&bslot0)[B0], uint16_t (&bslot1)[B1])
{
    constexpr bool WIDEN = FORM == kConvWiden, SPLIT = FORM == kConvSplit || WIDEN, HALF = FORM == kConvHalf;
    constexpr int CHUNKS = SPLIT? 4 : 2;  // weight transfers of a wave per stage
    constexpr int BM = 128, AV = 4;
    constexpr int PA = BM * kCRow;   // bf16 per A plane (80-byte rows)
    constexpr int PB = kCN * 32;     // bf16 per B plane (64-byte rows)
    // (opaque: values shared with the first try would sit in registers through its loop)
    int t = threadIdx.x;
    uint32_t tile_m = blockIdx.x;
    if constexpr (WIDEN) __asm__ volatile("" : "+v"(t), "+s"(tile_m));
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), lr = lane & 31, hh = lane >> 5;
    const int wm = wave & 1, wn = wave >> 1;
    const long long m0 = (long long)tile_m * BM;
    const int n0 = blockIdx.y * kCN;

    int iy0[AV], ix0[AV];
#pragma unroll
    for (int i = 0; i < AV; i++) {
        const long long m = m0 + t / 8 + 32 * i;
        if (m < a.M) {
            const uint32_t oy = (uint32_t)m / (uint32_t)a.OW, ox = (uint32_t)m - oy * (uint32_t)a.OW;
            iy0[i] = (int)oy * a.SY - a.PT;
            ix0[i] = (int)ox * a.SX - a.PL;
        } else {
            iy0[i] = -(1 << 30);
            ix0[i] = 0;
        }
    }
    // (stages counted from this piece's first: the whole inner range unless split)
    const int first = a.part? (int)blockIdx.z * a.piece_stages : 0;
    const int stages = a.part? min(a.piece_stages,a.Kp / kCK - first) : a.Kp / kCK;
    const uint32_t wbytes = (uint32_t)((size_t)a.Npad * a.Kp * 2);
    const CRsrc rx = conv_rsrc(a.x,(uint32_t)((size_t)a.W * a.H * a.C * 4));
    const CRsrc rwh = conv_rsrc(a.wh,wbytes), rwl = conv_rsrc(FORM == kConvSplit? a.wl : a.wh,wbytes);
    // B DMA: the stage's 16 (one plane: 8) chunks of 1 KB (plane c / 8, rows
    // 16 (c % 8) .. +15), chunk c = wave + 4i; lane l lands at row l / 4, physical piece l % 4
    uint32_t bvo[CHUNKS];
#pragma unroll
    for (int i = 0; i < CHUNKS; i++) {
        const int c = wave + 4 * i, row = 16 * (c % 8) + lane / 4, logical = (lane % 4) ^ ((row >> 2) & 3);
        bvo[i] = ((uint32_t)(n0 + row) * (uint32_t)a.Kp + 8u * (uint32_t)logical) * 2u;
    }
    auto issue_b = [&](int stage, int slot) {
#pragma unroll
        for (int i = 0; i < CHUNKS; i++) {
            const int c = wave + 4 * i;
            uint16_t* dst = (slot? bslot1 : bslot0) + (c / 8) * PB + (c % 8) * 512;
            conv_dma(c < 8? rwh : rwl,dst,bvo[i],(uint32_t)((first + stage) * kCK * 2));
        }
    };
    constexpr uint32_t kOut = 0x80000000u;
    uint32_t aoff[AV];
    int cur_tap = -1;
    auto fetch_a = [&](int stage, float4 (&ra)[AV]) {
        const int k0 = (first + stage) * kCK, tap = k0 / a.C;
        if (tap != cur_tap) {
            cur_tap = tap;
            const int ky = tap / a.KX, kx = tap % a.KX;
#pragma unroll
            for (int i = 0; i < AV; i++) {
                const int iy = iy0[i] + ky, ix = ix0[i] + kx;
                const bool in = iy >= 0 && iy < a.H && ix >= 0 && ix < a.W;
                const uint32_t pix = (uint32_t)iy * (uint32_t)a.W + (uint32_t)ix;
                aoff[i] = in? (pix * (uint32_t)a.C + (uint32_t)(t % 8) * 4u) * 4u : kOut;
            }
        }
        const uint32_t cb = (uint32_t)(k0 % a.C) * 4u;
#pragma unroll
        for (int i = 0; i < AV; i++) {
            const cu32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rx,aoff[i] + cb,0,0);
            ra[i] = make_float4(__uint_as_float(v.x),__uint_as_float(v.y),__uint_as_float(v.z),__uint_as_float(v.w));
        }
    };
    float top[HALF? AV : 1];  // largest |x| of this thread's share of each pixel's inputs
#pragma unroll
    for (int i = 0; i < (HALF? AV : 1); i++) top[i] = 0.0f;
    const float scale = probe.scale;
    auto store_a = [&](const float4 (&ra)[AV]) {
#pragma unroll
        for (int i = 0; i < AV; i++) {
            const int row = t / 8 + 32 * i, col = (t % 8) * 4;
            uint32_t h01, l01, h23, l23;
            if constexpr (HALF) {
                top[i] = __builtin_fmaxf(__builtin_fmaxf(top[i],__builtin_fabsf(ra[i].x)),__builtin_fabsf(ra[i].y));
                top[i] = __builtin_fmaxf(__builtin_fmaxf(top[i],__builtin_fabsf(ra[i].z)),__builtin_fabsf(ra[i].w));
                halves2_f16(ra[i].x,ra[i].y,scale,h01,l01);
                halves2_f16(ra[i].z,ra[i].w,scale,h23,l23);
            } else {
                halves2(ra[i].x,ra[i].y,h01,l01);
                halves2(ra[i].z,ra[i].w,h23,l23);
            }
            *reinterpret_cast<uint2*>(lds + row * kCRow + col) = make_uint2(h01,h23);
            *reinterpret_cast<uint2*>(lds + PA + row * kCRow + col) = make_uint2(l01,l23);
        }
    };

    v16f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = v16f{};
    auto multiply = [&](int slot) {
        const uint16_t* bs = slot? bslot1 : bslot0;
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            const int col = ks * 16 + 8 * hh;
            cu32x4 ah[2], al[2], bh[2], bl[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int row = wn * 64 + j * 32 + lr;
                const int at = row * 32 + (((2 * ks + hh) ^ ((row >> 2) & 3)) << 3);
                bh[j] = *reinterpret_cast<const cu32x4*>(bs + at);
                if constexpr (SPLIT) bl[j] = *reinterpret_cast<const cu32x4*>(bs + PB + at);
            }
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int row = wm * 64 + i * 32 + lr;
                ah[i] = *reinterpret_cast<const cu32x4*>(lds + row * kCRow + col);
                al[i] = *reinterpret_cast<const cu32x4*>(lds + PA + row * kCRow + col);
            }
            auto product = [](cu32x4 x, cu32x4 w, v16f c) {
                if constexpr (HALF) return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h,x),__builtin_bit_cast(v8h,w),c,0,0,0);
                else return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(cbf16x8,x),__builtin_bit_cast(cbf16x8,w),c,0,0,0);
            };
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    acc[i][j] = product(ah[i],bh[j],acc[i][j]);
                    if constexpr (SPLIT) acc[i][j] = product(ah[i],bl[j],acc[i][j]);
                    acc[i][j] = product(al[i],bh[j],acc[i][j]);
                }
        }
    };

    // Before stage s: A of s in LDS, B of s in slot s % 2, the loads of A of
    // s + 1 in flight in register set (s + 1) % 2.  Stage s issues B of s + 1
    // (the other slot, read last in stage s - 1) and A of s + 2 (set s % 2,
    // stored in stage s - 1), multiplies, and after a barrier waits for all
    // but the four newest loads (A of s + 2), so B of s + 1 and A of s + 1
    // have landed, and stores A of s + 1.
    if constexpr (WIDEN) {
        float4 ra[AV];
        for (int s = 0; s < stages; s++) {
            fetch_a(s,ra);
            // 128 rows x 64 bytes, two 16-byte pieces per thread
            cu32x4 rb[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int q = t + 256 * j;
                rb[j] = __builtin_amdgcn_raw_buffer_load_b128(rwh,(((uint32_t)n0 + q / 4) * (uint32_t)a.Kp + 8u * (q % 4)) * 2u,
                                                              (uint32_t)((first + s) * kCK * 2),0);
            }
            __syncthreads();  // every wave is done with the stage before
            store_a(ra);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int q = t + 256 * j, row = q / 4, at = row * 32 + (((q % 4) ^ ((row >> 2) & 3)) << 3);
                cu32x4 hi, lo;
                half_planes(rb[j],hi,lo);
                *reinterpret_cast<cu32x4*>(bslot0 + at) = hi;
                *reinterpret_cast<cu32x4*>(bslot0 + PB + at) = lo;
            }
            __syncthreads();
            multiply(0);
        }
    } else {
        float4 ra0[AV], ra1[AV];
        fetch_a(0,ra0);
        issue_b(0,0);
        // The image loads are issued unconditionally (past the last stage they
        // read offsets of a further tap, in range or read as zeros, and are never
        // stored), so every stage has the same four loads newest in the counter.
        fetch_a(1,ra1);
        store_a(ra0);
        conv_barrier<4>();  // B of 0 landed (A of 1 may be in flight)
        auto step = [&](int s, float4 (&mine)[AV], float4 (&next)[AV], int slot, bool more) {
            if (more) issue_b(s + 1,slot ^ 1);
            fetch_a(s + 2,mine);
            multiply(slot);
            if (more) {
                conv_barrier<15>();  // every wave is done reading A of s and B slot s % 2
                store_a(next);       // (the compiler waits for the loads of `next`)
                conv_barrier<4>();   // B of s + 1 landed; A of s + 2 may be in flight
            }
        };
        // Whole pairs in the loop (every step has a next stage, so the loop body
        // has no path that leaves a register set's loads unwaited), then the
        // last one or two stages.
        int s = 0;
        for (; s + 2 < stages; s += 2) {
            step(s,ra0,ra1,0,true);
            step(s + 1,ra1,ra0,1,true);
        }
        step(s,ra0,ra1,0,s + 1 < stages);
        if (s + 1 < stages) step(s + 1,ra1,ra0,1,false);
    }

    // A piece leaves its sums to conv_reduce_kernel, which adds the bias.
    float* const out = a.part? a.part + (size_t)blockIdx.z * (size_t)a.M * a.N : a.y;
    const float* const bias = a.part? nullptr : a.bias;
    float back = 1.0f;
    if constexpr (HALF) {
        // The pixels' maxima over the eight threads of each row.
        bool outside = false;
#pragma unroll
        for (int i = 0; i < AV; i++) {
            float m = top[i];
            m = __builtin_fmaxf(m,dpp_f32<kDppXor1>(m));
            m = __builtin_fmaxf(m,dpp_f32<kDppXor2>(m));
            m = __builtin_fmaxf(m,dpp_f32<kDppHalfMirror>(m));
            outside = outside || m * scale > 65504.0f || (m != 0.0f && (probe.blank >> i & 1));
        }
        if (__syncthreads_or(outside)) return true;
        back = 1.0f / scale;
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int n = n0 + wn * 64 + 32 * j + lr;
        if (n >= a.N) continue;
        const float b = bias? bias[n] : 0.0f;
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const long long m = m0 + wm * 64 + 32 * i + 8 * (r / 4) + 4 * hh + r % 4;
                const float v = HALF? acc[i][j][r] * back : acc[i][j][r];
                if (m < a.M) out[(size_t)m * a.N + n] = bias? __fadd_rn(v,b) : v;
            }
    }
    return false;
}

// The longer look and the second try are calls: inlined, their values take
// registers from the first try's loop.
typedef __attribute__((address_space(3))) uint8_t SharedBytes;
typedef const __attribute__((address_space(4))) ConvArgs KernelArgs;
__device__ __forceinline__ const ConvArgs& kernel_args(KernelArgs* args)
{
    const uint64_t p = (uint64_t)args;  // (the same in every lane)
    const uint64_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)p), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(p >> 32));
    return *(const ConvArgs*)(KernelArgs*)(lo | hi << 32);
}
__device__ __attribute__((noinline)) ConvProbe conv_longer_look(KernelArgs* args, SharedBytes* lds, SharedBytes* bslot0)
{
    return conv_probe<true>(kernel_args(args),(uint16_t*)(uint8_t*)lds,(uint16_t*)(uint8_t*)bslot0);
}
__device__ __attribute__((noinline)) void conv_second_try(KernelArgs* args, SharedBytes* lds, SharedBytes* bslot0, SharedBytes* bslot1)
{
    const ConvProbe probe = {1.0f,0};
    conv_body_ring<kConvWiden>(kernel_args(args),probe,*(uint16_t(*)[2 * 128 * kCRow])(uint8_t*)lds,
                               *(uint16_t(*)[2 * kCN * 32])(uint8_t*)bslot0,*(uint16_t(*)[kCN * 32])(uint8_t*)bslot1);
}

template <int FORM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3,3))) void conv_image_kernel(ConvArgs a)
{
    // (separate arrays: the compiler can then tell the image stores from the
    // transfers in flight into the ring)
    constexpr bool HALF = FORM == kConvHalf;
    __shared__ __attribute__((aligned(1024))) uint16_t lds[2 * 128 * kCRow];
    __shared__ __attribute__((aligned(1024))) uint16_t bslot0[2 * kCN * 32];  // ring slots: planes hi, lo
    __shared__ __attribute__((aligned(1024))) uint16_t bslot1[(FORM == kConvSplit? 2 : 1) * kCN * 32];
    ConvProbe probe = {1.0f,0};
    if constexpr (HALF) {
        auto args = (KernelArgs*)__builtin_amdgcn_kernarg_segment_ptr();
        auto *l = (SharedBytes*)(uint8_t*)lds, *b0 = (SharedBytes*)(uint8_t*)bslot0;
        probe = conv_probe<false>(a,lds,bslot0);
        if (probe.scale == 0.0f) {
            probe = conv_longer_look(args,l,b0);
            probe.scale = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(probe.scale)));
        }
        if (probe.scale == 0.0f || conv_body_ring<kConvHalf>(a,probe,lds,bslot0,bslot1))
            conv_second_try(args,l,b0,(SharedBytes*)(uint8_t*)bslot1);
    } else {
        conv_body_ring<FORM>(a,probe,lds,bslot0,bslot1);
    }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3,3))) void conv_image_wide_kernel(ConvArgs a)
{
    conv_body<1>(a);
}

__global__ __launch_bounds__(256) void conv_gather_kernel(ConvArgs a)
{
    conv_body<0>(a);
}

// y = the pieces' sums, in order, + bias.
__global__ __launch_bounds__(256) void conv_reduce_kernel(const float* __restrict__ part, int pieces, size_t total, int N, const float* bias,
                                                          float* __restrict__ y)
{
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= total) return;
    float v = part[e];
    for (int p = 1; p < pieces; p++) v += part[(size_t)p * total + e];
    y[e] = bias? __fadd_rn(v,bias[e % (unsigned)N]) : v;
}

// Whether a call runs the image kernel (a stage is whole channels, 32-bit offsets
// and pixels).
static bool image_form(const ConvArgs& a)
{
    const size_t lim = (size_t)1 << 31;
    return a.C % kCK == 0 && (reinterpret_cast<uintptr_t>(a.x) & 15) == 0 && (size_t)a.W * a.H * a.C * 4 < lim &&
           (size_t)a.Npad * a.Kp * 2 < lim && a.M < (long long)lim;
}

// Pieces of the inner range for images whose tiles leave CUs idle (one: none).
// A workgroup alone on a CU takes about 0.78 us a stage, several together 0.62
// each; pieces cost about 8 us more and a pass that moves (pieces + 1) fp32
// images at about 4 TB/s.  The estimate's least is taken.  Measured, us, whole /
// the pieces taken (F16 weights, 3x3): 40^2 pixels 512 -> 512 (52 tiles) 117.8 /
// 45, 64^2 (128 tiles) 118 / 70, 200 x 100 128 -> 3 (157 tiles) 36.5 / 27,
// 90^2 384 -> 384 (192 tiles) 92 / 80, 128^2 512 -> 256 (256 tiles) 120 / 117;
// 1x1 at 30^2 (16 stages) gains nothing and stays whole.  The prices are F16
// weights' for all: BF16 weights take as many products, F32 weights a quarter
// longer a stage, so that theirs stay whole a little longer than they should.
int conv_pieces(const ConvArgs& a)
{
    const long long tiles = (a.M + 127) / 128 * (a.Npad / kCN), cus = device_cus();
    const int stages = a.Kp / kCK;
    if (!image_form(a) || tiles > cus) return 1;
    int best = 1;
    double least = 0.78 * stages;
    for (int p = 2; p <= stages / 4 && p * tiles <= 3 * cus; p++) {
        const int length = (stages + p - 1) / p;
        if ((stages + length - 1) / length != p) continue;  // an empty last piece
        const long long rounds = (p * tiles + cus - 1) / cus;
        const double t = length * (rounds == 1? 0.78 : 0.62 * rounds) + 8.0 + (p + 1) * (double)a.M * a.N * 4.0 / 4e6;
        if (t < least) {
            least = t;
            best = p;
        }
    }
    return best;
}

hipError_t launch_conv(const ConvArgs& args, int pieces, float* part, hipStream_t s)
{
    ConvArgs a = args;
    if (!a.M || !a.N) return hipSuccess;
    const long long mt = (a.M + 127) / 128;
    if (mt > 0x7fffffffLL || a.Npad / kCN > 65535) return hipErrorInvalidValue;
    if (pieces > 1 && part) {
        a.part = part;
        a.piece_stages = (a.Kp / kCK + pieces - 1) / pieces;
    }
    const dim3 grid((unsigned)mt,(unsigned)(a.Npad / kCN),a.part? (unsigned)pieces : 1u);
    if (image_form(a)) {
        if (a.kind == kConvHalf) conv_image_kernel<kConvHalf><<<grid,dim3(256),0,s>>>(a);
        else if (a.kind == kConvBf16) conv_image_kernel<kConvBf16><<<grid,dim3(256),0,s>>>(a);
        else conv_image_kernel<kConvSplit><<<grid,dim3(256),0,s>>>(a);
    } else if (a.C % kCK == 0 && (reinterpret_cast<uintptr_t>(a.x) & 15) == 0) {
        conv_image_wide_kernel<<<grid,dim3(256),0,s>>>(a);
    } else {
        conv_gather_kernel<<<grid,dim3(256),0,s>>>(a);
    }
    if (a.part) {
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const size_t total = (size_t)a.M * a.N;
        conv_reduce_kernel<<<dim3((unsigned)((total + 255) / 256)),dim3(256),0,s>>>(part,pieces,total,a.N,a.bias,a.y);
    }
    return hipGetLastError();
}

}  // namespace pixhip
