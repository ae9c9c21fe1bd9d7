// denoise.hip -- BF16 3D U-Net fluence denoiser: MFMA implicit-GEMM
// convolution kernels (forward, data gradient, weight gradient), the
// pointwise layers, the loss, Adam, and the C-ABI of tam_denoise.h.
//
// Layout: activations are channels-last BF16, [z][y][x][c] (x fastest over
// voxels, c fastest overall); a 3x3x3 convolution with zero padding is the
// GEMM  Y[m][co] = sum_k X_im2col[m][k] W[k][co],  k = tap * Cin + ci,
// tap = 9 (dz+1) + 3 (dy+1) + (dx+1).  One v_mfma_f32_16x16x32_bf16 takes a
// 16-voxel x 32-k slab of X (lane l: voxel l%16, k 8 (l/16) .. +7, one
// 16-byte load of 8 consecutive channels) and a 32 x 16 slab of W (packed
// on the host side of each update into the lane order, one 16-byte load),
// and accumulates a 16 x 16 FP32 tile (lane l: voxels 4 (l/16) + j, output
// channel l%16).  Cin is a multiple of 16, so 8 consecutive k never cross
// a tap.
//
// The data gradient is the same kernel with the weights flipped in space and
// transposed (W'[26 - tap][co][ci]).  The weight gradient needs k = voxels:
// each wave stages 32 consecutive voxels of the layer input (shifted by one
// tap, zero outside) and of the output gradient in LDS, transposed to
// [channel][voxel], and reads 8 consecutive voxels of one channel per lane.
#include <cmath>
#include <cstring>
#include <new>
#include <random>
#include <string>
#include <vector>

#include "tam_internal.h"
#include "../../include/tam_denoise.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

__device__ __forceinline__ bf16x8 load8(const uint16_t* p) { return __builtin_bit_cast(bf16x8, *(const uint4*)p); }
__device__ __forceinline__ bf16x8 zero8() { return __builtin_bit_cast(bf16x8, make_uint4(0u, 0u, 0u, 0u)); }

struct ConvArgs {
    const uint16_t* x;      // input [nvox][cin]; with x2: the coarse grid [nvox / 8][c1]
    const uint16_t* wp;     // packed weights [kb][nt][64][8]
    const float* bias;      // [cout] or nullptr
    const uint16_t* mask;   // [nvox][cout] or nullptr: output *= (mask > 0)
    uint16_t* y;            // output [nvox][cout]
    int D, H, W, cin, cout, kb, relu;
    // input = cat(upsample2(x), x2) when x2 != nullptr: channels < c1 from the
    // coarse grid (nearest), the other cin - c1 from x2 [nvox][cin - c1]
    const uint16_t* x2;
    int c1;
};

// What the last convolution does with its result when nothing needs its
// activations afterwards: the head, and where `tally` is given the denoised
// tally from it.
struct HeadArgs {
    const uint16_t* x0;     // network input [nvox][4]
    const float* hw;        // 16 weights and the bias
    float* out;
    const float* mut;
    double nv;
    double* tally;
};

// head: x0[m][0] + hb + sum_c hw[c] a[m][c], a's 16 channels in u0 and u1
__device__ __forceinline__ float head_value(float first, const float* hw, const uint4& u0, const uint4& u1)
{
    float v = first + hw[16];
    const uint16_t* e0 = (const uint16_t*)&u0;
    const uint16_t* e1 = (const uint16_t*)&u1;
#pragma unroll
    for (int c = 0; c < 8; ++c) v += hw[c] * bf2f(e0[c]);
#pragma unroll
    for (int c = 0; c < 8; ++c) v += hw[8 + c] * bf2f(e1[c]);
    return v;
}

// the path length that the head's log1p(fluence) stands for; 0 in removed voxels
__device__ __forceinline__ double tally_value(float v, float mut, double nv)
{
    return mut > 0.f ? fmax(expm1((double)v), 0.0) * nv : 0.0;
}

// Raw buffer descriptor over `bytes` bytes from p (at most 2^31 - 1): loads
// at offsets past it return zero.  0x00020000: gfx9 buffer word 3 (32-bit
// data format, untyped access).
typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef unsigned v4u __attribute__((ext_vector_type(4)));
__device__ __forceinline__ Rsrc rsrc_n(const void* p, long bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(bytes < 0x7fffffffL ? bytes : 0x7fffffffL),
                                             0x00020000);
}
__device__ __forceinline__ bf16x8 bload8(Rsrc r, unsigned voff, unsigned soff)
{
    return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}

// Four consecutive channels co .. co + 3 of voxel m, out of cout: bias, ReLU
// and mask, one 8-byte store.  The convolutions give the weights to the MFMA
// as its rows and the voxels as its columns, so a lane holds four channels of
// one voxel and a wave's store covers whole 32-byte pieces of 16 voxels; with
// the voxels as rows it held one channel of four voxels, in four 2-byte stores
// (and loads of the mask).  The products and their order are the same.
__device__ __forceinline__ uint2 out4(const ConvArgs& a, const f32x4& acc, long m, int co, int cout)
{
    const float4 b = a.bias ? *(const float4*)(a.bias + co) : float4{0.f, 0.f, 0.f, 0.f};
    float v[4] = {acc[0] + b.x, acc[1] + b.y, acc[2] + b.z, acc[3] + b.w};
    uint2 mk = make_uint2(0u, 0u);
    if (a.mask) mk = *(const uint2*)(a.mask + m * cout + co);
    uint2 o;
    uint16_t* h = (uint16_t*)&o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (a.relu) v[j] = fmaxf(v[j], 0.f);
        if (a.mask && !(bf2f(((const uint16_t*)&mk)[j]) > 0.f)) v[j] = 0.f;
        h[j] = f2bf(v[j]);
    }
    return o;
}
__device__ __forceinline__ void store4(const ConvArgs& a, const f32x4& acc, long m, int co, int cout)
{
    *(uint2*)(a.y + m * cout + co) = out4(a, acc, m, co, cout);
}

// Convolutions of the quarter grid, whose x edge need not be a multiple of 16,
// and of 96 output channels: forward and, with flipped weights, data gradients.
// A wave computes 16 MT consecutive voxels of the flattened grid (each
// lane finds its voxel's x, y, z) for all NT x 16 output channels; CIN is
// the input channel count.
// Addressing: the input descriptor starts HW + W + 1 voxels before the
// block's first voxel, so every tap of the block's voxels sits at a
// non-negative 32-bit offset; a tap outside the grid (zero padding) gets an
// offset past the descriptor's end and loads zeros.  Each lane keeps a
// 27-bit mask of its voxel's valid taps.  With the k loop unrolled, a
// k-block's tap and channel for each of the four lane groups are constants,
// and their offsets scalar values.
template <int CIN, int NT>
__global__ __launch_bounds__(256) void conv_kernel(ConvArgs a)
{
    constexpr int MT = 4;
    constexpr int KB = (27 * CIN + 31) / 32;
    constexpr unsigned OUT = 0x80000000u;          // past every descriptor's end
    const int lane = threadIdx.x & 63, g = lane >> 4;
    const int W = a.W, H = a.H;
    const long HW = (long)H * W, nvox = HW * a.D;
    const long mblk = (long)blockIdx.x * (4 * 16 * MT);
    const long mbase = mblk + (long)(threadIdx.x >> 6) * (16 * MT);
    if (mbase >= nvox) return;
    const long back = HW + W + 1;
    const long vb = mblk > back ? mblk - back : 0;
    const Rsrc rx = rsrc_n(a.x + vb * CIN, (nvox - vb) * CIN * 2);
    const Rsrc rw = rsrc_n(a.wp, (long)KB * NT * 512 * 2);
    unsigned voff[MT], vmask[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const long m = mbase + t * 16 + (lane & 15);
        const int vx = (int)(m % W);
        const long r = m / W;
        const int vy = (int)(r % H), vz = (int)(r / H);
        voff[t] = (unsigned)((m - vb) * CIN * 2);
        const unsigned bx = (vx > 0 ? 1u : 0u) | 2u | (vx < W - 1 ? 4u : 0u);
        const unsigned by = (vy > 0 ? 1u : 0u) | 2u | (vy < H - 1 ? 4u : 0u);
        const unsigned bz = (vz > 0 ? 1u : 0u) | 2u | (vz < a.D - 1 ? 4u : 0u);
        unsigned vm = 0;
#pragma unroll
        for (int dz = 0; dz < 3; ++dz)
#pragma unroll
            for (int dy = 0; dy < 3; ++dy)
                if ((bz >> dz) & (by >> dy) & 1u) vm |= bx << (9 * dz + 3 * dy);
        vmask[t] = vm;
    }
    f32x4 acc[MT][NT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        // lane group gg holds k = 32 kb + 8 gg .. + 7: one tap, 8 channels
        int tapg[4], offg[4];
#pragma unroll
        for (int gg = 0; gg < 4; ++gg) {
            const int k = 32 * kb + 8 * gg;
            const int tap = k / CIN, ci = k % CIN;
            const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
            tapg[gg] = tap;                           // 27 (past the last tap) never has its mask bit set
            offg[gg] = (int)(((dz * HW + (long)dy * W + dx) * CIN + ci) * 2);
        }
        const int tap = g == 0 ? tapg[0] : g == 1 ? tapg[1] : g == 2 ? tapg[2] : tapg[3];
        const int toff = g == 0 ? offg[0] : g == 1 ? offg[1] : g == 2 ? offg[2] : offg[3];
        bf16x8 af[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const bool valid = (vmask[t] >> tap) & 1u;
            af[t] = bload8(rx, valid ? voff[t] + (unsigned)toff : OUT, 0);
        }
        bf16x8 bfr[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) bfr[n] = bload8(rw, (unsigned)lane * 16u, (unsigned)((kb * NT + n) * 1024));
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int n = 0; n < NT; ++n)
                acc[t][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[n], af[t], acc[t][n], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int n = 0; n < NT; ++n) store4(a, acc[t][n], mbase + t * 16 + (lane & 15), n * 16 + g * 4, NT * 16);
}

// Convolutions with at most 48 output channels, their input staged in LDS.
// In conv_kernel each A fragment of these layers feeds one or two MFMAs, so
// the vector-memory path, not the matrix cores, sets the rate.  Here a block
// computes an output brick of 16 (x) x 8 (y) x 4 (z) voxels.  For each group
// of 16 input channels it loads the input brick with a one-voxel halo
// (18 x 10 x 6 voxels x 16 channels, zeros outside the grid) into LDS, and
// every tap's A fragment is then an LDS read at a constant offset, with no
// per-tap validity test.  Wave w computes the 8 x-rows of plane z0 + w.  The
// k loop runs channel group by channel group (27 taps x 16 channels each, two
// taps per k-block), so each lane fetches its B fragment from the packed
// weights at that (tap, channel)'s place in their tap-major order.
// Grid edges must be multiples of 16 (x), 8 (y) and 4 (z); CIN a multiple of
// 16; NT = output channels / 16.
// 16 to 16 channels at 256^3: 459 us before the staging loads went out together
// and the stores held four channels, 336 after (1.07 GB: 3.2 of 5.2 TB/s); 48 to
// 16 1243, 977.  LDS reads take 110 us of the 336 and MFMAs 96; blocks that loop
// over bricks with the next brick's loads in flight were slower (367).
// FIRST: the first layer, whose input holds 4 of the 16 channels per voxel (8
// bytes to write and read instead of 32; the others are zero in LDS).
// HEAD: the last layer without a later backward pass; the output goes through
// LDS to the head instead of to memory and back (at 256^3 0.54 GB each way:
// 337 us, the head 228 and the tally 61 apart, 424 together).
enum { CONV_PLAIN, CONV_FIRST, CONV_HEAD };
template <int CIN, int NT, int KIND>
__global__ __launch_bounds__(256, NT == 1 ? 4 : CIN == 16 ? 2 : 3) void conv_lds_kernel(ConvArgs a, HeadArgs hd)
{
    constexpr bool FIRST = KIND == CONV_FIRST, HEAD = KIND == CONV_HEAD;
    constexpr int BX = 18, BY = 10, BZ = 6, CG = CIN / 16;
    constexpr int KB = (27 * CIN + 31) / 32;                  // k-blocks of the packed weights
    __shared__ __attribute__((aligned(16))) uint16_t sx[BZ * BY * BX * 16];
    const int W = a.W, H = a.H, D = a.D;
    const int gx = W / 16, gy = H / 8;
    // Workgroups go to the 8 XCDs in turn.  With several channel groups each XCD
    // takes one contiguous eighth of the bricks, whose shared halos then meet in
    // its L2 (48 channels at 256^3: 1040 us, 977; 96 at 128^3: 400, 382); one
    // group's input is read fastest in order (338, 347 the other way).
    const unsigned nb = gridDim.x;
    const unsigned bid = CG > 1 && nb % 8 == 0 ? blockIdx.x % 8 * (nb / 8) + blockIdx.x / 8 : blockIdx.x;
    const int bxi = bid % gx, byi = (bid / gx) % gy, bzi = bid / (gx * gy);
    const int x0 = bxi * 16, y0 = byi * 8, z0 = bzi * 4;
    const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const Rsrc rw = rsrc_n(a.wp, (long)KB * NT * 512 * 2);
    f32x4 acc[8][NT];
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int cg = 0; cg < CG; ++cg) {
        if (cg > 0) __syncthreads();                          // the previous group's reads are done
        // Stage channels 16 cg .. 16 cg + 15 of the input brick, 16-byte chunks,
        // two per voxel: all of a thread's loads first, then its LDS writes.
        // (One load at a time, each waiting for the last, was most of the
        // kernel.)  A load of a wave takes the 16 inner voxels of two rows: its
        // base is a scalar, its lane offsets are constants, and rows outside
        // the grid read zeros past the descriptor's end.
        {
            const bool cat = a.x2 != nullptr, coarse = cat && 16 * cg < a.c1;
            const uint16_t* src = cat && !coarse ? a.x2 : a.x;
            const int sh = coarse ? 1 : 0, sc = !cat ? (FIRST ? 4 : CIN) : coarse ? a.c1 : CIN - a.c1;
            const int c0 = cat && !coarse ? 16 * cg - a.c1 : 16 * cg;
            const int Ws = W >> sh, Hs = H >> sh;
            const int row = lane >> 5, lx = (lane & 31) >> 1, half = lane & 1;
            const unsigned off = (unsigned)(((row * Ws + (lx >> sh)) * sc + half * 8) * 2);
            constexpr unsigned OUT = 0x80000000u;                 // past every descriptor's end
            constexpr int PAIRS = BZ * BY / 2;                    // row pairs; wave w takes w, w + 4, ..
            bf16x8 v[(PAIRS + 3) / 4], vh = zero8();
#pragma unroll
            for (int i = 0; i < (PAIRS + 3) / 4; ++i) {
                const int p = min(w + 4 * i, PAIRS - 1), lz = p / (BY / 2), ly = p % (BY / 2) * 2;
                const int yy = y0 - 1 + ly, zz = z0 - 1 + lz;      // rows yy and yy + 1 of plane zz
                const uint16_t* base =
                    src + (((long)(zz >> sh) * Hs + (yy >> sh)) * Ws + (x0 >> sh)) * sc + c0;
                const Rsrc rs = rsrc_n(base, zz >= 0 && zz < D ? 0x7fffffffL : 0L);
                const bool outside = (yy < 0 && row == 0) || (yy + 1 >= H && row == 1);
                if constexpr (FIRST) {
                    typedef unsigned v2u __attribute__((ext_vector_type(2)));
                    const v2u q = __builtin_amdgcn_raw_buffer_load_b64(rs, outside || half ? (int)OUT : (int)off, 0, 0);
                    v[i] = __builtin_bit_cast(bf16x8, make_uint4(q.x, q.y, 0u, 0u));
                } else {
                    v[i] = bload8(rs, outside ? OUT : off, 0);
                }
            }
            // the columns beside them: a chunk a thread
            const int hr = (int)threadIdx.x >> 2, side = ((int)threadIdx.x >> 1) & 1;
            if (threadIdx.x < BZ * BY * 4) {
                const int xx = side ? x0 + 16 : x0 - 1, yy = y0 - 1 + hr % BY, zz = z0 - 1 + hr / BY;
                if (xx >= 0 && xx < W && yy >= 0 && yy < H && zz >= 0 && zz < D) {
                    const long at = (((long)(zz >> sh) * Hs + (yy >> sh)) * Ws + (xx >> sh)) * sc + c0;
                    if constexpr (FIRST) {
                        const uint2 u = half ? make_uint2(0u, 0u) : *(const uint2*)(src + at);
                        vh = __builtin_bit_cast(bf16x8, make_uint4(u.x, u.y, 0u, 0u));
                    } else {
                        vh = load8(src + at + half * 8);
                    }
                }
            }
            uint16_t* dst = sx + ((w * 2 + row) * BX + 1 + lx) * 16 + half * 8;
#pragma unroll
            for (int i = 0; i < (PAIRS + 3) / 4; ++i)
                if (w + 4 * i < PAIRS) *(bf16x8*)(dst + i * 8 * BX * 16) = v[i];
            if (threadIdx.x < BZ * BY * 4) *(bf16x8*)(sx + (hr * BX + side * 17) * 16 + half * 8) = vh;
        }
        __syncthreads();
        // k-block kb: lane group g takes tap 2 kb + g / 2, channels 16 cg +
        // 8 (g % 2) .. + 7.  Tap 27 (the last block's second half) is the
        // packed weights' zero padding (or past the descriptor's end, which
        // reads zeros): its A fragment repeats tap 26, a finite value times 0.
        auto load = [&](int kb, bf16x8* af, bf16x8* bfr) {
            const int tapr = 2 * kb + (g >> 1), ci0 = 8 * (g & 1);
            const int tap = tapr < 27 ? tapr : 26;
            const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
            const int base = ((w + dz + 1) * BY + (dy + 1)) * BX + (r + dx + 1);
#pragma unroll
            for (int t = 0; t < 8; ++t) af[t] = *(const bf16x8*)(sx + (base + t * BX) * 16 + ci0);
            // this lane's k in the packed (tap-major) order: its k-block and lane group there
            const int ko = tapr * CIN + 16 * cg + ci0;
            const int kbo = ko >> 5, go = (ko >> 3) & 3;
#pragma unroll
            for (int n = 0; n < NT; ++n)
                bfr[n] = bload8(rw, (unsigned)((go * 16 + r) * 16), (unsigned)((kbo * NT + n) * 1024));
        };
        auto mma = [&](const bf16x8* af, const bf16x8* bfr) {
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    acc[t][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[n], af[t], acc[t][n], 0, 0, 0);
        };
        // two fragment sets in turn: the next k-block's reads are in flight
        // while the current one's MFMAs run
        bf16x8 afa[8], bfa[NT], afb[8], bfb[NT];
        load(0, afa, bfa);
        if constexpr (CG == 1 && NT == 1) {
            // unrolled: the accumulators stay in place (in a loop the compiler
            // rotates them through one register quad every iteration)
#pragma unroll
            for (int kb = 0; kb < 14; kb += 2) {
                load(kb + 1, afb, bfb);
                mma(afa, bfa);
                if (kb + 2 < 14) load(kb + 2, afa, bfa);
                mma(afb, bfb);
            }
        } else {
            // rolled: unrolled, the wider kernels grow past 160 VGPRs, and the
            // channel-group loop copies the accumulators anyway
#pragma unroll 1
            for (int kb = 0; kb < 14; kb += 2) {
                load(kb + 1, afb, bfb);
                mma(afa, bfa);
                if (kb + 2 < 14) load(kb + 2, afa, bfa);
                mma(afb, bfb);
            }
        }
    }
    if constexpr (HEAD) {
        __syncthreads();                                      // the input's reads are done
#pragma unroll
        for (int t = 0; t < 8; ++t)
            *(uint2*)(sx + ((w * 8 + t) * 16 + r) * 16 + g * 4) = out4(a, acc[t][0], 0, g * 4, 16);
        __syncthreads();
        for (int q = threadIdx.x; q < 512; q += 256) {
            const long m = ((long)(z0 + (q >> 7)) * H + (y0 + ((q >> 4) & 7))) * W + x0 + (q & 15);
            const float v = head_value(bf2f(hd.x0[m * 4]), hd.hw, *(const uint4*)(sx + q * 16),
                                       *(const uint4*)(sx + q * 16 + 8));
            if (hd.tally) hd.tally[m] = tally_value(v, hd.mut[m], hd.nv);
            else hd.out[m] = v;
        }
    } else {
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int n = 0; n < NT; ++n)
                store4(a, acc[t][n], ((long)(z0 + w) * H + (y0 + t)) * W + x0 + r, n * 16 + g * 4, NT * 16);
    }
}

struct WgradArgs {
    const uint16_t* x;      // layer input [nvox][cin]
    const uint16_t* dy;     // output gradient [nvox][cout]
    float* gw;              // [27][cin][cout], accumulated with atomics
    int D, H, W, cin, cout;
    long blocks;            // 32-voxel segments of the flattened grid
    long per_wg;            // segments per workgroup (a multiple of 4)
};

// Weight gradient for one tap (blockIdx.y) over a range of 32-voxel
// segments (blockIdx.x): dW^T[co][ci] += sum_m dy[m][co] x[m + tap][ci].
template <int CIT, int COT>
__global__ __launch_bounds__(256) void wgrad_kernel(WgradArgs a)
{
    constexpr int CI = CIT * 16, CO = COT * 16;
    constexpr int PAD = 8;                                  // row pad (elements) against bank conflicts
    __shared__ __attribute__((aligned(16))) uint16_t sX[4][CI][32 + PAD];
    __shared__ __attribute__((aligned(16))) uint16_t sD[4][CO][32 + PAD];
    __shared__ float sR[CI * CO];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int tap = blockIdx.y;
    const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
    f32x4 acc[COT][CIT];
#pragma unroll
    for (int i = 0; i < COT; ++i)
#pragma unroll
        for (int c = 0; c < CIT; ++c) acc[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    const long b0 = (long)blockIdx.x * a.per_wg;
    const long b1 = b0 + a.per_wg < a.blocks ? b0 + a.per_wg : a.blocks;
    for (long bb = b0; bb < b1; bb += 4) {
        const long blk = bb + wv;
        const bool have = blk < b1;
        if (have) {
            // segment blk: the 32 consecutive voxels 32 blk .. 32 blk + 31 of
            // the flattened grid (each finds its own x, y, z below)
            const long mrow = blk * 32;
            // dy: 32 voxels x CO channels, 8 channels per lane-load
            for (int q = lane; q < 32 * CO / 8; q += 64) {
                const int v = q / (CO / 8), c8 = (q % (CO / 8)) * 8;
                const uint4 d = *(const uint4*)(a.dy + (mrow + v) * a.cout + c8);
                const uint16_t* e = (const uint16_t*)&d;
#pragma unroll
                for (int j = 0; j < 8; ++j) sD[wv][c8 + j][v] = e[j];
            }
            // x shifted by the tap, zero outside the grid
            for (int q = lane; q < 32 * CI / 8; q += 64) {
                const int v = q / (CI / 8), c8 = (q % (CI / 8)) * 8;
                const long m = mrow + v;
                const int x = (int)(m % a.W);
                const long r = m / a.W;
                const int sx = x + dx, sy = (int)(r % a.H) + dy, sz = (int)(r / a.H) + dz;
                uint4 d = make_uint4(0u, 0u, 0u, 0u);
                if (sx >= 0 && sx < a.W && sy >= 0 && sy < a.H && sz >= 0 && sz < a.D)
                    d = *(const uint4*)(a.x + (((long)sz * a.H + sy) * a.W + sx) * a.cin + c8);
                const uint16_t* e = (const uint16_t*)&d;
#pragma unroll
                for (int j = 0; j < 8; ++j) sX[wv][c8 + j][v] = e[j];
            }
        }
        __syncthreads();
        if (have) {
            const int k8 = (lane >> 4) * 8, r16 = lane & 15;
            bf16x8 bx[CIT];
#pragma unroll
            for (int c = 0; c < CIT; ++c) bx[c] = load8(&sX[wv][c * 16 + r16][k8]);
#pragma unroll
            for (int i = 0; i < COT; ++i) {
                const bf16x8 ad = load8(&sD[wv][i * 16 + r16][k8]);
#pragma unroll
                for (int c = 0; c < CIT; ++c)
                    acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ad, bx[c], acc[i][c], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // reduce the four waves in LDS, then one atomic per weight
    for (int q = threadIdx.x; q < CI * CO; q += 256) sR[q] = 0.f;
    __syncthreads();
    for (int w = 0; w < 4; ++w) {
        if (wv == w) {
#pragma unroll
            for (int i = 0; i < COT; ++i)
#pragma unroll
                for (int c = 0; c < CIT; ++c)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int co = i * 16 + (lane >> 4) * 4 + j, ci = c * 16 + (lane & 15);
                        sR[ci * CO + co] += acc[i][c][j];
                    }
        }
        __syncthreads();
    }
    for (int q = threadIdx.x; q < CI * CO; q += 256)
        if (sR[q] != 0.f) atomicAdd(&a.gw[(long)tap * CI * CO + q], sR[q]);
}

// Weight gradient by output bricks, all of a 16-channel input tile's taps at
// once: dW^T[co][ci] += sum_m dy[m][co] x[m + tap][ci].
//
// A block stages a 16 (x) x 8 (y) x 4 (z) brick of dy (COT x 16 channels) and
// the matching 18 x 10 x 6 brick of x (one 16-channel tile, zeros outside the
// grid), both transposed to [channel][voxel] in LDS, once per brick.  Wave w
// owns plane w of the brick: four 32-voxel k-chunks (row pairs), whose dy
// fragments stay in registers while it walks the taps.  Per chunk and (dz, dy)
// one aligned 8-voxel x read plus two dwords give the dx = -1, 0, +1 fragments
// (v_alignbyte), so one LDS read feeds 3 x COT MFMAs.  NDZ = 1: the block
// covers all 27 taps; NDZ = 3: the 9 taps of one dz (blockIdx.y % 3).
// blockIdx.y / NDZ is the input-channel tile.  At 128^3, 16 to 16 channels:
// 121 us with the staging loads one after the other, 81 with all of them first
// and one round of blocks; 32 outputs 82, 47.  The products alone take 53 and 27.
// Blocks loop over bricks and
// keep their sums in registers; at the end the four waves are summed in LDS
// and each block writes its partial [taps][16][CO] to `part`, which
// wgradb_reduce_kernel sums into gw.  The blocks of grid row 0 also sum dy
// over their bricks (the bias gradient, CO floats after the weights).
struct WgradbArgs {
    const uint16_t* x;      // layer input [nvox][cin]; with x2: the coarse grid [nvox / 8][c1]
    const uint16_t* dy;     // output gradient [nvox][cout]
    float* part;            // [gridDim.y][gridDim.x]: [taps][16][cout] weights, then [cout] bias
    int D, H, W, cin, cout;
    long bricks;            // (W / 16) (H / 8) (D / 4)
    const uint16_t* x2;     // input = cat(upsample2(x), x2) when not null (see ConvArgs)
    int c1;
};

// FIRST: the first layer's input, 4 of the 16 channels per voxel.
template <int COT, int NDZ, bool FIRST>
__global__ __launch_bounds__(256) void wgradb_kernel(WgradbArgs a)
{
    constexpr int CO = COT * 16, NT = 27 / NDZ;
    constexpr int XR = 24;                                  // x row: element 4 + v holds voxel x0 + v (v = -1 .. 16)
    constexpr int XC = 6 * 10 * XR + 4;                     // x channel stride (elements), padded against bank conflicts
    constexpr int DC = 4 * 8 * 16 + 8;                      // dy channel stride (elements), padded likewise
    constexpr int NW = NT * 16 * CO;                       // weights per partial
    constexpr int XBYTES = 16 * XC * 2, DBYTES = CO * DC * 2, RBYTES = (NW + CO) * 4;
    constexpr int LBYTES = (XBYTES + DBYTES > RBYTES ? XBYTES + DBYTES : RBYTES);
    __shared__ __attribute__((aligned(16))) unsigned char lds[LBYTES];
    uint16_t* sX = (uint16_t*)lds;
    uint16_t* sD = (uint16_t*)(lds + XBYTES);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int r16 = lane & 15, g = lane >> 4, h = g & 1, gr = g >> 1;
    const int ct = (int)blockIdx.y / NDZ;                   // input-channel tile
    const int dz0 = NDZ == 1 ? -1 : (int)blockIdx.y % 3 - 1;
    const int W = a.W, H = a.H, D = a.D;
    const int bx = W / 16, by = H / 8;
    f32x4 acc[NT][COT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < COT; ++i) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bool bias = blockIdx.y == 0;
    float bsum[COT];
#pragma unroll
    for (int i = 0; i < COT; ++i) bsum[i] = 0.f;

    // Staging.  x: voxel pairs (x0 + 2p, x0 + 2p + 1), p = 0 .. 7, of 10 rows x 6
    // planes (4 where the block does one dz), 16 channels as two 8-channel
    // halves; each lane loads both voxels' half and writes one dword (the pair)
    // per channel; then the columns beside them, a voxel's half a thread.  dy:
    // voxel pairs of 16 x 8 x 4 voxels, CO channels in 8-channel groups.  All
    // loads of a brick go out before its first write (an item at a time, seven
    // waits for memory came one after the other); outside the grid x reads the
    // tensor's first voxel and counts as zeros.
    constexpr int ROWS = NDZ == 1 ? 60 : 40, NI = (ROWS * 16 + 255) / 256, ND = CO / 8;
    const int lz0 = NDZ == 1 ? 0 : dz0 + 1;                 // first plane of the x brick that is needed
    const bool cat = a.x2 != nullptr, coarse = cat && ct * 16 < a.c1;
    const uint16_t* xs = cat && !coarse ? a.x2 : a.x;
    const int sh = coarse ? 1 : 0, sc = !cat ? (FIRST ? 4 : a.cin) : coarse ? a.c1 : a.cin - a.c1;
    const int c0 = cat && !coarse ? ct * 16 - a.c1 : ct * 16;
    const int half = threadIdx.x & 1, pp = ((int)threadIdx.x >> 1) & 7;
    const int hr = (int)threadIdx.x >> 2, side = ((int)threadIdx.x >> 1) & 1;
    const bool halo = threadIdx.x < ROWS * 4;
    uint4 v0[NI], v1[NI], vh, d0[ND], d1[ND];
    bool in[NI];
    auto fetch = [&](long b) {
        const int x0 = (int)(b % bx) * 16, y0 = (int)((b / bx) % by) * 8, z0 = (int)(b / ((long)bx * by)) * 4;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int row = min(((int)threadIdx.x >> 4) + 16 * i, ROWS - 1);   // the last rows twice, alike
            const int yy = y0 - 1 + row % 10, zz = z0 - 1 + lz0 + row / 10;
            in[i] = yy >= 0 && yy < H && zz >= 0 && zz < D;
            const long vr = ((long)(zz >> sh) * (H >> sh) + (yy >> sh)) * (W >> sh);
            const long at = in[i] ? (vr + ((x0 + 2 * pp) >> sh)) * sc : 0;
            if constexpr (FIRST) {                           // 4 channels a voxel, the pair in 16 bytes
                v0[i] = *(const uint4*)(xs + at);
            } else {
                const uint16_t* q = xs + at + c0 + half * 8;
                v0[i] = *(const uint4*)q;
                v1[i] = *(const uint4*)(q + (coarse ? 0 : sc));
            }
        }
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            const int q = (int)threadIdx.x + 256 * i, vq = 2 * (q / ND), c8 = (q % ND) * 8;
            const int lx = vq & 15, ly = (vq >> 4) & 7, lz = vq >> 7;
            const uint16_t* src = a.dy + (((long)(z0 + lz) * H + (y0 + ly)) * W + (x0 + lx)) * a.cout + c8;
            d0[i] = *(const uint4*)src;
            d1[i] = *(const uint4*)(src + a.cout);
        }
        vh = make_uint4(0u, 0u, 0u, 0u);
        if (halo) {
            const int xx = side ? x0 + 16 : x0 - 1, yy = y0 - 1 + hr % 10, zz = z0 - 1 + lz0 + hr / 10;
            if (xx >= 0 && xx < W && yy >= 0 && yy < H && zz >= 0 && zz < D) {
                const uint16_t* q = xs + (((long)(zz >> sh) * (H >> sh) + (yy >> sh)) * (W >> sh) + (xx >> sh)) * sc + c0;
                if constexpr (FIRST) {
                    const uint2 u = half ? make_uint2(0u, 0u) : *(const uint2*)q;
                    vh = make_uint4(u.x, u.y, 0u, 0u);
                } else {
                    vh = *(const uint4*)(q + half * 8);
                }
            }
        }
    };
    auto commit = [&] {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int row = min(((int)threadIdx.x >> 4) + 16 * i, ROWS - 1);
            if constexpr (FIRST) {
                v1[i] = make_uint4(v0[i].z, v0[i].w, 0u, 0u);
                v0[i] = make_uint4(v0[i].x, v0[i].y, 0u, 0u);
                in[i] = in[i] && half == 0;
            }
            if (!in[i]) v0[i] = v1[i] = make_uint4(0u, 0u, 0u, 0u);
            const uint16_t* e0 = (const uint16_t*)&v0[i];
            const uint16_t* e1 = (const uint16_t*)&v1[i];
            uint16_t* dst = sX + (half * 8) * XC + (lz0 * 10 + row) * XR + 4 + 2 * pp;
#pragma unroll
            for (int j = 0; j < 8; ++j) *(uint32_t*)(dst + j * XC) = (uint32_t)e0[j] | ((uint32_t)e1[j] << 16);
        }
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            const int q = (int)threadIdx.x + 256 * i, vq = 2 * (q / ND), c8 = (q % ND) * 8;
            const uint16_t* e0 = (const uint16_t*)&d0[i];
            const uint16_t* e1 = (const uint16_t*)&d1[i];
            uint16_t* dst = sD + c8 * DC + vq;
#pragma unroll
            for (int j = 0; j < 8; ++j) *(uint32_t*)(dst + j * DC) = (uint32_t)e0[j] | ((uint32_t)e1[j] << 16);
        }
        if (halo) {
            const uint16_t* e = (const uint16_t*)&vh;
            uint16_t* dst = sX + (half * 8) * XC + (lz0 * 10 + hr) * XR + (side ? 20 : 3);
#pragma unroll
            for (int j = 0; j < 8; ++j) dst[j * XC] = e[j];
        }
    };
    // (The next brick's loads in flight during a brick's products gave nothing,
    // 48 us against 47 for 32 outputs: two blocks a CU already overlap.)
    for (long b = blockIdx.x; b < a.bricks; b += gridDim.x) {
        fetch(b);
        __syncthreads();                                    // the last brick's reads are done
        commit();
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            // dy^T fragment of chunk c: channel r16 of tile i, voxels 8h .. 8h + 7 of row 2c + gr, plane wv
            bf16x8 ad[COT];
#pragma unroll
            for (int i = 0; i < COT; ++i) ad[i] = load8(sD + (i * 16 + r16) * DC + (wv * 8 + 2 * c + gr) * 16 + 8 * h);
            if (bias) {
#pragma unroll
                for (int i = 0; i < COT; ++i)
#pragma unroll
                    for (int j = 0; j < 8; ++j) bsum[i] += (float)ad[i][j];
            }
            // all of the chunk's x reads first (one wait for the lot), then its MFMAs
            constexpr int NR = (NDZ == 1 ? 3 : 1) * 3;
            uint2 m0[NR], m1[NR];
            unsigned prev[NR], next[NR];
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                // x row of channel r16 at plane wv + dz, row 2c + gr + dy (halo coordinates +1)
                const int dz = dz0 + r / 3, ky = r % 3;
                const uint16_t* row = sX + r16 * XC + ((wv + dz + 1) * 10 + (2 * c + gr + ky)) * XR;
                m0[r] = *(const uint2*)(row + 4 + 8 * h);                       // voxels 8h .. 8h + 3
                m1[r] = *(const uint2*)(row + 8 + 8 * h);                       // voxels 8h + 4 .. 8h + 7
                prev[r] = *(const unsigned*)(row + 2 + 8 * h);                  // high half: voxel 8h - 1
                next[r] = *(const unsigned*)(row + 12 + 8 * h);                 // low half: voxel 8h + 8
            }
#pragma unroll
            for (int kz = 0; kz < (NDZ == 1 ? 3 : 1); ++kz) {
#pragma unroll
                for (int ky = 0; ky < 3; ++ky) {
                    const int r = kz * 3 + ky;
                    uint4 mid, lo, hi;
                    mid.x = m0[r].x; mid.y = m0[r].y; mid.z = m1[r].x; mid.w = m1[r].y;
                    lo.x = __builtin_amdgcn_alignbyte(mid.x, prev[r], 2);
                    lo.y = __builtin_amdgcn_alignbyte(mid.y, mid.x, 2);
                    lo.z = __builtin_amdgcn_alignbyte(mid.z, mid.y, 2);
                    lo.w = __builtin_amdgcn_alignbyte(mid.w, mid.z, 2);
                    hi.x = __builtin_amdgcn_alignbyte(mid.y, mid.x, 2);
                    hi.y = __builtin_amdgcn_alignbyte(mid.z, mid.y, 2);
                    hi.z = __builtin_amdgcn_alignbyte(mid.w, mid.z, 2);
                    hi.w = __builtin_amdgcn_alignbyte(next[r], mid.w, 2);
                    const bf16x8 bx3[3] = {__builtin_bit_cast(bf16x8, lo), __builtin_bit_cast(bf16x8, mid),
                                           __builtin_bit_cast(bf16x8, hi)};
#pragma unroll
                    for (int kx = 0; kx < 3; ++kx)
#pragma unroll
                        for (int i = 0; i < COT; ++i) {
                            const int t = (kz * 3 + ky) * 3 + kx;
                            acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ad[i], bx3[kx], acc[t][i], 0, 0, 0);
                        }
                }
            }
        }
    }
    // the four waves' sums: wave 0 stores, the others add in turn; then the
    // block's partial goes out (element (t, ci, co) at (t * 16 + ci) * CO + co)
    float* sR = (float*)lds;
    __syncthreads();                                        // the last brick's reads are done
    for (int w = 0; w < 4; ++w) {
        if (wv == w) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < COT; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int q = (t * 16 + r16) * CO + i * 16 + 4 * g + j;
                        sR[q] = (w == 0 ? 0.f : sR[q]) + acc[t][i][j];
                    }
        }
        __syncthreads();
    }
    // bias: the four k-groups of a channel, then the waves in turn
#pragma unroll
    for (int i = 0; i < COT; ++i) {
        bsum[i] += __shfl_xor(bsum[i], 16, 64);
        bsum[i] += __shfl_xor(bsum[i], 32, 64);
    }
    for (int w = 0; w < 4; ++w) {
        if (wv == w && g == 0) {
#pragma unroll
            for (int i = 0; i < COT; ++i) sR[NW + i * 16 + r16] = (w == 0 ? 0.f : sR[NW + i * 16 + r16]) + bsum[i];
        }
        __syncthreads();
    }
    float* out = a.part + ((long)blockIdx.y * gridDim.x + blockIdx.x) * (NW + CO);
    for (int q = threadIdx.x; q < NW + CO; q += 256) out[q] = sR[q];
}

// gw[tap][ci][co] += the sum over the nb blocks of one blockIdx.y of their
// partials; ny rows of blocks, ndz dz groups per input-channel tile.  Block
// column blockIdx.y of this grid sums partials k = blockIdx.y, blockIdx.y +
// gridDim.y, ... and adds its share atomically, so a weight sums over enough
// blocks in parallel to hide the memory latency.
__global__ __launch_bounds__(256) void wgradb_reduce_kernel(const float* __restrict__ part, int nb, int ny, int ndz,
                                                            int cin, int cout, float* __restrict__ gw,
                                                            float* __restrict__ gb)
{
    const int nt = 27 / ndz;
    const long nw = (long)nt * 16 * cout, per = nw + cout;
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    if (q >= per * ny) return;
    const int yrow = (int)(q / per);
    const long e = q % per;
    if (e >= nw && yrow != 0) return;                       // only grid row 0 sums the bias
    const float* src = part + (long)yrow * nb * per + e;
    float s = 0.f;
    for (int k = (int)blockIdx.y; k < nb; k += (int)gridDim.y) s += src[(long)k * per];
    if (e >= nw) {
        atomicAdd(&gb[e - nw], s);
        return;
    }
    const int t = (int)(e / (16 * cout)), ci = (int)((e / cout) % 16), co = (int)(e % cout);
    const int ct = yrow / ndz, tap = (ndz == 1 ? 0 : (yrow % 3) * 9) + t;
    atomicAdd(&gw[((long)tap * cin + ct * 16 + ci) * cout + co], s);
}

// bias gradient: gb[c] += sum_m d[m][c], c a multiple of 8 (<= 2048); each lane reads 8 channels of a voxel
__global__ __launch_bounds__(256) void bgrad_kernel(const uint16_t* d, long nvox, int c, float* gb)
{
    __shared__ float s[256 * 8];
    const int g = c / 8, per = 256 / g;                     // 8-channel groups per voxel, voxels per pass
    const int cg = threadIdx.x % g, vi = threadIdx.x / g;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (vi < per)
        for (long m = (long)blockIdx.x * per + vi; m < nvox; m += (long)gridDim.x * per) {
            const uint4 u = *(const uint4*)(d + m * c + cg * 8);
            const uint16_t* e = (const uint16_t*)&u;
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] += bf2f(e[j]);
        }
#pragma unroll
    for (int j = 0; j < 8; ++j) s[threadIdx.x * 8 + j] = acc[j];
    __syncthreads();
    for (int ch = threadIdx.x; ch < c; ch += 256) {
        float t = 0.f;
        for (int v = 0; v < per; ++v) t += s[(v * g + ch / 8) * 8 + ch % 8];
        atomicAdd(&gb[ch], t);
    }
}

// The pointwise layers move 8 consecutive BF16 channels (16 bytes) per
// thread: every channel count here is a multiple of 8, so a chunk never
// straddles two source tensors.
struct Bf8 {
    uint16_t h[8];
};
__device__ __forceinline__ Bf8 ld8(const uint16_t* p) { return __builtin_bit_cast(Bf8, *(const uint4*)p); }
__device__ __forceinline__ void st8(uint16_t* p, const Bf8& v) { *(uint4*)p = __builtin_bit_cast(uint4, v); }

// 2x2x2 average pooling; one thread per coarse voxel and 8-channel chunk
__global__ void pool_kernel(const uint16_t* x, int D, int H, int W, int C, uint16_t* y)
{
    const int C8 = C / 8, Wc = W / 2, Hc = H / 2;
    const long n = (long)(D / 2) * Hc * Wc * C8;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        const int c = (int)(q % C8) * 8;
        long r = q / C8;
        const int xo = (int)(r % Wc); r /= Wc;
        const int yo = (int)(r % Hc);
        const int zo = (int)(r / Hc);
        float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < 8; ++k) {
            const int xi = 2 * xo + (k & 1), yi = 2 * yo + ((k >> 1) & 1), zi = 2 * zo + (k >> 2);
            const Bf8 v = ld8(x + (((long)zi * H + yi) * W + xi) * C + c);
#pragma unroll
            for (int j = 0; j < 8; ++j) s[j] += bf2f(v.h[j]);
        }
        Bf8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o.h[j] = f2bf(0.125f * s[j]);
        st8(y + q * 8, o);
    }
}

// gradient of the upsampled part of a concatenation, summed onto the coarse
// grid and masked by the coarse ReLU output: d[mc][c] = (sum of the 8
// children's g[child][c]) * (a[mc][c] > 0), c < C1; one thread per coarse
// voxel and 8-channel chunk
__global__ void upcat_bwd_kernel(const uint16_t* g, int C, int C1, const uint16_t* a, int D, int H, int W,
                                 uint16_t* d)
{
    const int Dc = D / 2, Hc = H / 2, Wc = W / 2, C18 = C1 / 8;
    const long n = (long)Dc * Hc * Wc * C18;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        const int c = (int)(q % C18) * 8;
        long r = q / C18;
        const int xc = (int)(r % Wc); r /= Wc;
        const int yc = (int)(r % Hc);
        const int zc = (int)(r / Hc);
        float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < 8; ++k) {
            const int x = 2 * xc + (k & 1), yy = 2 * yc + ((k >> 1) & 1), z = 2 * zc + (k >> 2);
            const Bf8 v = ld8(g + (((long)z * H + yy) * W + x) * C + c);
#pragma unroll
            for (int j = 0; j < 8; ++j) s[j] += bf2f(v.h[j]);
        }
        const Bf8 av = ld8(a + q * 8);
        Bf8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) o.h[j] = bf2f(av.h[j]) > 0.f ? f2bf(s[j]) : (uint16_t)0;
        st8(d + q * 8, o);
    }
}

// gradient of a ReLU output that feeds a skip connection and a pooling:
// d[m][c] = (g_cat[m][C1 + c] + g_pool[parent(m)][c] / 8) * (a[m][c] > 0);
// one thread per fine voxel and 8-channel chunk
__global__ void skip_pool_bwd_kernel(const uint16_t* gcat, int Ccat, int C1, const uint16_t* gpool,
                                     const uint16_t* a, int D, int H, int W, int C, uint16_t* d)
{
    const int C8 = C / 8;
    const long n = (long)D * H * W * C8;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        const int c = (int)(q % C8) * 8;
        const long m = q / C8;
        const int x = (int)(m % W);
        const long r = m / W;
        const int yy = (int)(r % H), z = (int)(r / H);
        const long mp = ((long)(z / 2) * (H / 2) + yy / 2) * (W / 2) + x / 2;
        const Bf8 gc = ld8(gcat + m * Ccat + C1 + c), gp = ld8(gpool + mp * C + c), av = ld8(a + q * 8);
        Bf8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float sj = bf2f(gc.h[j]) + 0.125f * bf2f(gp.h[j]);
            o.h[j] = bf2f(av.h[j]) > 0.f ? f2bf(sj) : (uint16_t)0;
        }
        st8(d + q * 8, o);
    }
}

// features (4 x nvox FP32) -> the network's input, 4 BF16 channels a voxel
__global__ void pack_input_kernel(const float* f, long nvox, uint16_t* x0)
{
    for (long m = (long)blockIdx.x * blockDim.x + threadIdx.x; m < nvox; m += (long)gridDim.x * blockDim.x) {
        uint2 o;
        uint16_t* v = (uint16_t*)&o;
        for (int c = 0; c < 4; ++c) v[c] = f2bf(f[(long)c * nvox + m]);
        *(uint2*)(x0 + m * 4) = o;
    }
}

// features from a context: phi = L / (npk V), mu_a and mu_s from mu_t and
// the material's albedo
__global__ void ctx_features_kernel(const double* tally, const float* mut, const uint8_t* mat,
                                    const MatEntry* mtab, long nvox, double inv_nv, float* f)
{
    for (long m = (long)blockIdx.x * blockDim.x + threadIdx.x; m < nvox; m += (long)gridDim.x * blockDim.x) {
        const float mu = mut[m], alb = mtab[mat[m]].albedo;
        const float mua = mu * (1.f - alb), mus = mu * alb;
        f[m] = (float)log1p(tally[m] * inv_nv);
        f[nvox + m] = log10f(fmaxf(mua, 1e-3f));
        f[2 * nvox + m] = log10f(fmaxf(mus, 1e-2f)) - 2.f;
        f[3 * nvox + m] = 5.f * (mtab[mat[m]].g - 0.8f);
    }
}

// the same features written straight into the BF16 input (the
// forward-only path: no FP32 staging)
__global__ void ctx_input_kernel(const double* tally, const float* mut, const uint8_t* mat, const MatEntry* mtab,
                                 long nvox, double inv_nv, uint16_t* x0)
{
    for (long m = (long)blockIdx.x * blockDim.x + threadIdx.x; m < nvox; m += (long)gridDim.x * blockDim.x) {
        const float mu = mut[m], alb = mtab[mat[m]].albedo;
        const float mua = mu * (1.f - alb), mus = mu * alb;
        uint2 o;
        uint16_t* v = (uint16_t*)&o;
        // round to FP32 first, as the staged path stores it: the empty asm keeps
        // the compiler from folding double -> float -> BF16 into one rounding
        float l = (float)log1p(tally[m] * inv_nv);
        asm volatile("" : "+v"(l));
        v[0] = f2bf(l);
        v[1] = f2bf(log10f(fmaxf(mua, 1e-3f)));
        v[2] = f2bf(log10f(fmaxf(mus, 1e-2f)) - 2.f);
        v[3] = f2bf(5.f * (mtab[mat[m]].g - 0.8f));
        *(uint2*)(x0 + m * 4) = o;
    }
}

// features (4 x nvox FP32) + target log1p(phi_hi) from a context -> slot
__global__ void store_slot_kernel(const float* f, const double* tally_hi, double inv_nv_hi, long nvox,
                                  uint16_t* feat, float* tgt)
{
    for (long m = (long)blockIdx.x * blockDim.x + threadIdx.x; m < nvox; m += (long)gridDim.x * blockDim.x) {
        for (int c = 0; c < 4; ++c) feat[m * 4 + c] = f2bf(f[(long)c * nvox + m]);
        tgt[m] = tally_hi ? (float)log1p(tally_hi[m] * inv_nv_hi) : f[4 * nvox + m];
    }
}

// head of a training step: out[m], and its L1 against an FP32 target with the
// loss summed into *loss (the input's into *base)
__global__ __launch_bounds__(256) void head_kernel(const uint16_t* x0, const uint16_t* a, const float* hw,
                                                   long nvox, float* out, const float* tgt, double* loss,
                                                   double* base)
{
    __shared__ double s[2][256];
    double l = 0.0, lb = 0.0;
    for (long m = (long)blockIdx.x * 256 + threadIdx.x; m < nvox; m += (long)gridDim.x * 256) {
        const float first = bf2f(x0[m * 4]);
        const float v = head_value(first, hw, *(const uint4*)(a + m * 16), *(const uint4*)(a + m * 16 + 8));
        out[m] = v;
        const float t = tgt[m];
        l += fabsf(v - t);
        lb += fabsf(first - t);
    }
    s[0][threadIdx.x] = l;
    s[1][threadIdx.x] = lb;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            s[0][threadIdx.x] += s[0][threadIdx.x + o];
            s[1][threadIdx.x] += s[1][threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        atomicAdd(loss, s[0][0]);
        if (base) atomicAdd(base, s[1][0]);
    }
}

// head backward: g = sign(out - t) / nvox; d9[m][c] = g hw[c] (a > 0);
// ghw[c] += sum g a[m][c]; ghw[16] += sum g
__global__ __launch_bounds__(256) void head_bwd_kernel(const float* out, const float* tgt, const uint16_t* a,
                                                       const float* hw, long nvox, uint16_t* d9, float* ghw)
{
    __shared__ float s[17][256];
    float acc[17];
    for (int c = 0; c < 17; ++c) acc[c] = 0.f;
    const float inv = 1.f / (float)nvox;
    for (long m = (long)blockIdx.x * 256 + threadIdx.x; m < nvox; m += (long)gridDim.x * 256) {
        const float diff = out[m] - tgt[m];
        const float g = (diff > 0.f ? inv : (diff < 0.f ? -inv : 0.f));
        uint4 u[2] = {*(const uint4*)(a + m * 16), *(const uint4*)(a + m * 16 + 8)};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint16_t* e = (uint16_t*)&u[h];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int c = 8 * h + j;
                const float av = bf2f(e[j]);
                acc[c] += g * av;
                e[j] = av > 0.f ? f2bf(g * hw[c]) : (uint16_t)0;
            }
            *(uint4*)(d9 + m * 16 + 8 * h) = u[h];
        }
        acc[16] += g;
    }
    for (int c = 0; c < 17; ++c) s[c][threadIdx.x] = acc[c];
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o)
            for (int c = 0; c < 17; ++c) s[c][threadIdx.x] += s[c][threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x < 17) atomicAdd(&ghw[threadIdx.x], s[threadIdx.x][0]);
}

// Adam on the FP32 parameter vector
__global__ void adam_kernel(float* p, const float* g, float* m1, float* m2, long n, float lr, float b1, float b2,
                            float c1, float c2, float eps)
{
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        const float gq = g[q];
        const float a = b1 * m1[q] + (1.f - b1) * gq;
        const float b = b2 * m2[q] + (1.f - b2) * gq * gq;
        m1[q] = a;
        m2[q] = b;
        p[q] -= lr * (a * c1) / (sqrtf(b * c2) + eps);
    }
}

// pack FP32 W[27][cin][cout] into MFMA B fragments: [kb][nt][lane][8],
// element (kb, nt, lane, j) = W at k = 32 kb + 8 (lane/16) + j, co = 16 nt +
// lane%16.  flip: the data-gradient weights W'[26 - tap][co][ci] (cin and
// cout swap roles).
__device__ __forceinline__ void pack_w(const float* w, int cin, int cout, int flip, int kb_n, uint16_t* wp)
{
    const int ci_eff = flip ? cout : cin, co_eff = flip ? cin : cout;
    const int nt = co_eff / 16;
    const long n = (long)kb_n * nt * 64 * 8;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) {
        const int j = (int)(q % 8);
        long r = q / 8;
        const int lane = (int)(r % 64); r /= 64;
        const int t = (int)(r % nt);
        const int kb = (int)(r / nt);
        const int k = kb * 32 + (lane >> 4) * 8 + j;
        const int tap = k / ci_eff, ci = k % ci_eff, co = t * 16 + (lane & 15);
        float v = 0.f;
        if (tap < 27) v = flip ? w[((long)(26 - tap) * cin + co) * cout + ci] : w[((long)tap * cin + ci) * cout + co];
        wp[q] = f2bf(v);
    }
}

// every layer's forward and data-gradient packing in one launch: grid row
// blockIdx.y packs job y (rows past a small job's extent exit at once)
struct PackJob {
    const float* w;
    uint16_t* wp;
    int cin, cout, flip, kb_n;
};
constexpr int kPackJobs = 20;           // two per layer (the network's ten layers)
struct PackJobs {
    PackJob j[kPackJobs];
};
__global__ void pack_all_kernel(PackJobs jobs)
{
    const PackJob& J = jobs.j[blockIdx.y];
    pack_w(J.w, J.cin, J.cout, J.flip, J.kb_n, J.wp);
}

__global__ void fill_f32k(float* p, long n, float v)
{
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) p[q] = v;
}
__global__ void fill_f64k(double* p, long n, double v)
{
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x) p[q] = v;
}

unsigned grid_of(long n, int per = 256)
{
    long b = (n + per - 1) / per;
    if (b > 16384) b = 16384;
    return (unsigned)(b < 1 ? 1 : b);
}

// ---------------------------------------------------------------- network --

struct Layer {
    int cin, cout, level;       // level 0: full grid, 1: /2, 2: /4
    long w_off, b_off;          // offsets in the parameter vector
    int kb_f, kb_b;             // k blocks of the forward / data-gradient GEMM
    uint16_t *wf, *wb;          // packed BF16 weights
};

constexpr int NL = 10;
static_assert(2 * NL == kPackJobs, "one forward and one data-gradient packing per layer");
constexpr int CIN[NL] = {16, 16, 16, 32, 32, 64, 96, 32, 48, 16};
constexpr int COUT[NL] = {16, 16, 32, 32, 64, 64, 32, 32, 16, 16};
constexpr int LEVEL[NL] = {0, 0, 1, 1, 2, 2, 1, 1, 0, 0};

}  // namespace

struct tam_dn {
    int dev, ncu;
    hipStream_t stream;
    hipEvent_t ev0, ev1;
    std::string err;
    int D[3], H[3], W[3];
    long nv[3];
    Layer L[NL];
    long nparam, head_off;
    float *p, *g, *m1, *m2;           // parameters, gradients, Adam moments
    long step;
    // activations (BF16) and their gradients
    uint16_t *x0, *a[NL], *p1, *p3;
    uint16_t *d[NL], *gc6, *gc8, *gp1, *gp3;
    float *out, *feat;                // FP32 head output; FP32 feature staging (5 x nvox)
    float* wpart;                     // per-block weight-gradient partials of the brick kernel
    long wpart_n;                     // its size in floats
    double* red;                      // [0] loss, [1] input loss
    // dataset
    int capacity;
    uint16_t* ds_feat;                // [slot][nvox][4] BF16 features
    float* ds_tgt;                    // [slot][nvox] FP32 target log(1 + phi_hi)
    float last_ms;
};

namespace {

int dfail(tam_dn* n, int code, const std::string& m)
{
    if (n) n->err = m;
    return code;
}
#define DNCHK(n, call)                                                                      \
    do {                                                                                    \
        hipError_t e_ = (call);                                                             \
        if (e_ != hipSuccess) return dfail((n), TAM_ERR_HIP, std::string(#call ": ") + hipGetErrorString(e_)); \
    } while (0)

thread_local std::string g_dn_err;

hipError_t conv_launch(tam_dn* n, const uint16_t* x, int lvl, int cin, const uint16_t* wp, int kb, const float* bias,
                       int cout, int relu, const uint16_t* mask, uint16_t* y, const uint16_t* x2 = nullptr,
                       int c1 = 0, int c4 = 0, const HeadArgs* head = nullptr)
{
    ConvArgs a{x, wp, bias, mask, y, n->D[lvl], n->H[lvl], n->W[lvl], cin, cout, kb, relu, x2, c1};
    const long nv = n->nv[lvl];
    // conv_kernel's blocks are 4 waves of 64 voxels; every level's voxel count is
    // a multiple of 512
    if (nv % 512 != 0 || kb != (27 * cin + 31) / 32) return hipErrorInvalidValue;
    const unsigned nb = (unsigned)(nv / (4 * 64));
#define CV(CI, NT_) hipLaunchKernelGGL((conv_kernel<CI, NT_>), dim3(nb), dim3(256), 0, n->stream, a)
    const int D = n->D[lvl], H = n->H[lvl], W = n->W[lvl];
    if (W % 16 == 0 && H % 8 == 0 && D % 4 == 0) {
        // LDS-staged input for up to 48 output channels from 16 (at 128^3 107 us
        // against 157 with the input read by each fragment); 64 outputs of the
        // coarse levels are faster without (32^3: 49 us against 65)
        const dim3 grid((unsigned)((W / 16) * (H / 8) * (D / 4)));
#define CL(CI, NT_) hipLaunchKernelGGL((conv_lds_kernel<CI, NT_, CONV_PLAIN>), grid, dim3(256), 0, n->stream, a, HeadArgs{})
        if (head || c4) {
            if (cin != 16 || cout != 16 || (head && c4)) return hipErrorInvalidValue;
            if (head)
                hipLaunchKernelGGL((conv_lds_kernel<16, 1, CONV_HEAD>), grid, dim3(256), 0, n->stream, a, *head);
            else
                hipLaunchKernelGGL((conv_lds_kernel<16, 1, CONV_FIRST>), grid, dim3(256), 0, n->stream, a, HeadArgs{});
            return hipGetLastError();
        }
        switch (cin * 1000 + cout) {
        case 16016: CL(16, 1); return hipGetLastError();
        case 16032: CL(16, 2); return hipGetLastError();
        case 16048: CL(16, 3); return hipGetLastError();
        case 32032: CL(32, 2); return hipGetLastError();
        case 96032: CL(96, 2); return hipGetLastError();
        case 48016: CL(48, 1); return hipGetLastError();
        case 32016: CL(32, 1); return hipGetLastError();
        }
#undef CL
    }
    // read or done by the LDS form only, which every other layer takes: the full
    // and the half grid's edges are multiples of 32 and 16
    if (x2 || c4 || head) return hipErrorInvalidValue;
    switch (cin * 1000 + cout) {
    case 32064: CV(32, 4); break; // layer 4
    case 64064: CV(64, 4); break; // layer 5 and its data gradient
    case 64032: CV(64, 2); break; // data gradient of layer 4
    case 32096: CV(32, 6); break; // data gradient of layer 6
    default: return hipErrorInvalidValue;
    }
#undef CV
    return hipGetLastError();
}

// The brick weight-gradient launch of a layer: grid rows (input-channel
// tiles x dz groups), dz groups, blocks per row and partial floats per block;
// false where the layer keeps the segment kernels (grid edges not multiples of
// 16 / 8 / 4).
struct BrickPlan {
    int ny, ndz;
    long nb, per;
};
bool brick_plan(int ncu, int D, int H, int W, int cin, int cout, BrickPlan* bp)
{
    if (W % 16 != 0 || H % 8 != 0 || D % 4 != 0 || cin % 16 != 0) return false;
    if (cout != 16 && cout != 32 && cout != 64) return false;
    bp->ndz = cout == 16 ? 1 : 3;                          // all 27 taps' sums in registers when they fit
    bp->ny = (cin / 16) * bp->ndz;
    const long bricks = (long)(W / 16) * (H / 8) * (D / 4);
    // one round of resident blocks (their LDS lets a CU hold two, of 64 output
    // channels one), with the same number of bricks each: at 128^3 16 to 16
    // channels 85 us with 1024 blocks, 78; 64 outputs 44, 36; the partials' sum
    // 9.4, 5.8
    long nb = (long)ncu * (cout == 64 ? 1 : 2) / bp->ny;
    if (nb < 1) nb = 1;
    const long each = (bricks + nb - 1) / nb;
    bp->nb = (bricks + each - 1) / each;
    bp->per = (27 / bp->ndz) * 16L * cout + cout;
    return true;
}

}  // namespace

extern "C" int64_t tam_internal_brick_blocks(int ncu, int D, int H, int W, int cin, int cout)
{
    BrickPlan bp;
    return brick_plan(ncu, D, H, W, cin, cout, &bp) ? bp.nb * bp.ny : 0;
}

namespace {

// weight gradient of one layer into gw; the brick form also sums the bias
// gradient into gb and says so in *bias_done
hipError_t wgrad_launch(tam_dn* n, const uint16_t* x, const uint16_t* dy, int lvl, int cin, int cout, float* gw,
                        float* gb, bool* bias_done, const uint16_t* x2 = nullptr, int c1 = 0, int c4 = 0)
{
    *bias_done = false;
    BrickPlan bp;
    if (brick_plan(n->ncu, n->D[lvl], n->H[lvl], n->W[lvl], cin, cout, &bp) && n->wpart &&
        (long)bp.ny * bp.nb * bp.per <= n->wpart_n) {
        WgradbArgs b{x, dy, n->wpart, n->D[lvl], n->H[lvl], n->W[lvl], cin, cout,
                     (long)(n->W[lvl] / 16) * (n->H[lvl] / 8) * (n->D[lvl] / 4), x2, c1};
        const dim3 grid((unsigned)bp.nb, (unsigned)bp.ny);
        if (c4 && cout != 16) return hipErrorInvalidValue;
        if (c4) hipLaunchKernelGGL((wgradb_kernel<1, 1, true>), grid, dim3(256), 0, n->stream, b);
        else if (cout == 16) hipLaunchKernelGGL((wgradb_kernel<1, 1, false>), grid, dim3(256), 0, n->stream, b);
        else if (cout == 32) hipLaunchKernelGGL((wgradb_kernel<2, 3, false>), grid, dim3(256), 0, n->stream, b);
        else hipLaunchKernelGGL((wgradb_kernel<4, 3, false>), grid, dim3(256), 0, n->stream, b);
        // ~1024 reduction blocks: each weight's nb partials split over ksplit of them
        const unsigned qb = grid_of(bp.ny * bp.per);
        long ks = 1024 / (long)qb;
        if (ks < 1) ks = 1;
        if (ks > bp.nb) ks = bp.nb;
        hipLaunchKernelGGL(wgradb_reduce_kernel, dim3(qb, (unsigned)ks), dim3(256), 0, n->stream, n->wpart,
                           (int)bp.nb, bp.ny, bp.ndz, cin, cout, gw, gb);
        *bias_done = true;
        return hipGetLastError();
    }
    if (x2 || c4) return hipErrorInvalidValue;  // read by the brick form only
    // one workgroup per tap and range of segments, ~96 per tap
    WgradArgs a{x, dy, gw, n->D[lvl], n->H[lvl], n->W[lvl], cin, cout, 0, 0};
    a.blocks = n->nv[lvl] / 32;
    long per = (a.blocks + 95) / 96;
    per = (per + 3) / 4 * 4;
    if (per < 4) per = 4;
    a.per_wg = per;
    const dim3 grid((unsigned)((a.blocks + per - 1) / per), 27);
    // the layers of the quarter grid, whose x edge may be an odd multiple of 8
    if (cin == 32 && cout == 64) hipLaunchKernelGGL((wgrad_kernel<2, 4>), grid, dim3(256), 0, n->stream, a);
    else if (cin == 64 && cout == 64) hipLaunchKernelGGL((wgrad_kernel<4, 4>), grid, dim3(256), 0, n->stream, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t repack(tam_dn* n)
{
    PackJobs jobs;
    unsigned gx = 1;
    for (int l = 0; l < NL; ++l) {
        const Layer& L = n->L[l];
        const float* w = n->p + L.w_off;
        jobs.j[2 * l] = PackJob{w, L.wf, L.cin, L.cout, 0, L.kb_f};
        jobs.j[2 * l + 1] = PackJob{w, L.wb, L.cin, L.cout, 1, L.kb_b};
        gx = std::max(gx, grid_of((long)L.kb_f * L.cout * 32));
        gx = std::max(gx, grid_of((long)L.kb_b * L.cin * 32));
    }
    hipLaunchKernelGGL(pack_all_kernel, dim3(gx, kPackJobs), dim3(256), 0, n->stream, jobs);
    return hipGetLastError();
}

// forward from the input x0 ([nvox][4]).  With tgt: activations kept for
// backward(), the prediction in n->out and the L1 loss summed into red[0]
// (input's in red[1]).  Without: the prediction in n->out, or with c the
// denoised tally in c (nv: packets times the voxel volume).
hipError_t forward(tam_dn* n, const uint16_t* x0, const float* tgt, tam_ctx* c = nullptr, double nv = 0.0)
{
    hipError_t e;
    auto conv = [&](int l, const uint16_t* in, uint16_t* o) {
        const Layer& L = n->L[l];
        return conv_launch(n, in, L.level, L.cin, L.wf, L.kb_f, n->p + L.b_off, L.cout, 1, nullptr, o);
    };
    const Layer& L0 = n->L[0];
    if ((e = conv_launch(n, x0, L0.level, L0.cin, L0.wf, L0.kb_f, n->p + L0.b_off, L0.cout, 1, nullptr, n->a[0], nullptr,
                         0, 1)) != hipSuccess)
        return e;
    if ((e = conv(1, n->a[0], n->a[1])) != hipSuccess) return e;
    hipLaunchKernelGGL(pool_kernel, dim3(grid_of(n->nv[1] * 16 / 8)), dim3(256), 0, n->stream, n->a[1], n->D[0], n->H[0],
                       n->W[0], 16, n->p1);
    if ((e = conv(2, n->p1, n->a[2])) != hipSuccess) return e;
    if ((e = conv(3, n->a[2], n->a[3])) != hipSuccess) return e;
    hipLaunchKernelGGL(pool_kernel, dim3(grid_of(n->nv[2] * 32 / 8)), dim3(256), 0, n->stream, n->a[3], n->D[1], n->H[1],
                       n->W[1], 32, n->p3);
    if ((e = conv(4, n->p3, n->a[4])) != hipSuccess) return e;
    if ((e = conv(5, n->a[4], n->a[5])) != hipSuccess) return e;
    // layers 6 and 8 read cat(upsample2(coarse), skip) in their input staging
    auto conv_cat = [&](int l, const uint16_t* coarse, int c1, const uint16_t* skip, uint16_t* o) {
        const Layer& L = n->L[l];
        return conv_launch(n, coarse, L.level, L.cin, L.wf, L.kb_f, n->p + L.b_off, L.cout, 1, nullptr, o, skip, c1);
    };
    if ((e = conv_cat(6, n->a[5], 64, n->a[3], n->a[6])) != hipSuccess) return e;
    if ((e = conv(7, n->a[6], n->a[7])) != hipSuccess) return e;
    if ((e = conv_cat(8, n->a[7], 32, n->a[1], n->a[8])) != hipSuccess) return e;
    if (!tgt) {
        const HeadArgs h{x0, n->p + n->head_off, n->out, c ? c->mut : nullptr, nv, c ? c->tally : nullptr};
        const Layer& L9 = n->L[9];
        return conv_launch(n, n->a[8], L9.level, L9.cin, L9.wf, L9.kb_f, n->p + L9.b_off, L9.cout, 1, nullptr, nullptr,
                           nullptr, 0, 0, &h);
    }
    if ((e = conv(9, n->a[8], n->a[9])) != hipSuccess) return e;
    hipLaunchKernelGGL(fill_f64k, dim3(1), dim3(64), 0, n->stream, n->red, 2L, 0.0);
    // every workgroup ends in atomics onto two addresses: at most 1024 workgroups
    const unsigned hg = grid_of(n->nv[0]);
    hipLaunchKernelGGL(head_kernel, dim3(hg > 1024u ? 1024u : hg), dim3(256), 0, n->stream, x0, n->a[9],
                       n->p + n->head_off, n->nv[0], n->out, tgt, n->red, n->red + 1);
    return hipGetLastError();
}

// backward after forward(x0, tgt): gradients of the mean L1 into n->g
hipError_t backward(tam_dn* n, const uint16_t* x0, const float* tgt)
{
    hipError_t e;
    hipLaunchKernelGGL(fill_f32k, dim3(grid_of(n->nparam)), dim3(256), 0, n->stream, n->g, n->nparam, 0.f);
    const unsigned hb = grid_of(n->nv[0]) < 1024u ? grid_of(n->nv[0]) : 1024u;
    hipLaunchKernelGGL(head_bwd_kernel, dim3(hb), dim3(256), 0, n->stream, n->out, tgt, n->a[9],
                       n->p + n->head_off, n->nv[0], n->d[9], n->g + n->head_off);
    auto grads = [&](int l, const uint16_t* in, const uint16_t* dl, const uint16_t* x2 = nullptr, int c1 = 0,
                     int c4 = 0) {
        const Layer& L = n->L[l];
        bool bias_done = false;
        hipError_t r = wgrad_launch(n, in, dl, L.level, L.cin, L.cout, n->g + L.w_off, n->g + L.b_off, &bias_done,
                                    x2, c1, c4);
        if (r != hipSuccess || bias_done) return r;
        // at most 1024 blocks: every block ends in `cout` atomics onto the same few addresses, which serialise
        if (L.cout % 8 != 0 || L.cout > 2048) return hipErrorInvalidValue;
        unsigned nb = grid_of(n->nv[L.level], 256 / (L.cout / 8));
        hipLaunchKernelGGL(bgrad_kernel, dim3(nb < 1024u ? nb : 1024u), dim3(256), 0, n->stream, dl,
                           n->nv[L.level], L.cout, n->g + L.b_off);
        return hipGetLastError();
    };
    // data gradient of layer l into `o`, masked by `mask` (the ReLU output feeding l), if any
    auto dgrad = [&](int l, const uint16_t* dl, const uint16_t* mask, uint16_t* o) {
        const Layer& L = n->L[l];
        return conv_launch(n, dl, L.level, L.cout, L.wb, L.kb_b, nullptr, L.cin, 0, mask, o);
    };
    if ((e = grads(9, n->a[8], n->d[9])) != hipSuccess) return e;
    if ((e = dgrad(9, n->d[9], n->a[8], n->d[8])) != hipSuccess) return e;
    if ((e = grads(8, n->a[7], n->d[8], n->a[1], 32)) != hipSuccess) return e;
    if ((e = dgrad(8, n->d[8], nullptr, n->gc8)) != hipSuccess) return e;
    hipLaunchKernelGGL(upcat_bwd_kernel, dim3(grid_of(n->nv[1] * 32 / 8)), dim3(256), 0, n->stream, n->gc8, 48, 32,
                       n->a[7], n->D[0], n->H[0], n->W[0], n->d[7]);
    if ((e = grads(7, n->a[6], n->d[7])) != hipSuccess) return e;
    if ((e = dgrad(7, n->d[7], n->a[6], n->d[6])) != hipSuccess) return e;
    if ((e = grads(6, n->a[5], n->d[6], n->a[3], 64)) != hipSuccess) return e;
    if ((e = dgrad(6, n->d[6], nullptr, n->gc6)) != hipSuccess) return e;
    hipLaunchKernelGGL(upcat_bwd_kernel, dim3(grid_of(n->nv[2] * 64 / 8)), dim3(256), 0, n->stream, n->gc6, 96, 64,
                       n->a[5], n->D[1], n->H[1], n->W[1], n->d[5]);
    if ((e = grads(5, n->a[4], n->d[5])) != hipSuccess) return e;
    if ((e = dgrad(5, n->d[5], n->a[4], n->d[4])) != hipSuccess) return e;
    if ((e = grads(4, n->p3, n->d[4])) != hipSuccess) return e;
    if ((e = dgrad(4, n->d[4], nullptr, n->gp3)) != hipSuccess) return e;
    hipLaunchKernelGGL(skip_pool_bwd_kernel, dim3(grid_of(n->nv[1] * 32 / 8)), dim3(256), 0, n->stream, n->gc6, 96, 64,
                       n->gp3, n->a[3], n->D[1], n->H[1], n->W[1], 32, n->d[3]);
    if ((e = grads(3, n->a[2], n->d[3])) != hipSuccess) return e;
    if ((e = dgrad(3, n->d[3], n->a[2], n->d[2])) != hipSuccess) return e;
    if ((e = grads(2, n->p1, n->d[2])) != hipSuccess) return e;
    if ((e = dgrad(2, n->d[2], nullptr, n->gp1)) != hipSuccess) return e;
    hipLaunchKernelGGL(skip_pool_bwd_kernel, dim3(grid_of(n->nv[0] * 16 / 8)), dim3(256), 0, n->stream, n->gc8, 48, 32,
                       n->gp1, n->a[1], n->D[0], n->H[0], n->W[0], 16, n->d[1]);
    if ((e = grads(1, n->a[0], n->d[1])) != hipSuccess) return e;
    if ((e = dgrad(1, n->d[1], n->a[0], n->d[0])) != hipSuccess) return e;
    if ((e = grads(0, x0, n->d[0], nullptr, 0, 1)) != hipSuccess) return e;
    return hipGetLastError();
}

hipError_t adam(tam_dn* n, float lr)
{
    ++n->step;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f / (1.f - std::pow(b1, (float)n->step));
    const float c2 = 1.f / (1.f - std::pow(b2, (float)n->step));
    hipLaunchKernelGGL(adam_kernel, dim3(grid_of(n->nparam)), dim3(256), 0, n->stream, n->p, n->g, n->m1, n->m2,
                       n->nparam, lr, b1, b2, c1, c2, 1e-8f);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return repack(n);
}

struct DevScope {
    int prev = -1;
    explicit DevScope(int d)
    {
        hipGetDevice(&prev);
        if (prev != d) hipSetDevice(d);
    }
    ~DevScope()
    {
        int cur = -1;
        hipGetDevice(&cur);
        if (prev >= 0 && cur != prev) hipSetDevice(prev);
    }
};

float ms_between(tam_dn* n)
{
    float ms = 0.f;
    hipEventElapsedTime(&ms, n->ev0, n->ev1);
    return ms;
}

}  // namespace

extern "C" {

int tam_dn_create(int32_t device, int32_t nx, int32_t ny, int32_t nz, int32_t capacity, uint64_t seed, tam_dn** out)
{
    if (!out) return TAM_ERR_ARG;
    *out = nullptr;
    if (nx < 32 || ny < 32 || nz < 32 || nx % 32 || ny % 32 || nz % 32 || capacity < 0) {
        g_dn_err = "grid edges must be positive multiples of 32";
        return TAM_ERR_ARG;
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
        g_dn_err = "no HIP device";
        return TAM_ERR_NODEVICE;
    }
    if (device < 0 || device >= ndev) {
        g_dn_err = "device ordinal out of range";
        return TAM_ERR_ARG;
    }
    tam_dn* n = new (std::nothrow) tam_dn();
    if (!n) return TAM_ERR_NOMEM;
    n->dev = device;
    DevScope ds(device);
    n->ncu = mc_device().ncu;
    for (int l = 0; l < 3; ++l) {
        n->W[l] = nx >> l;
        n->H[l] = ny >> l;
        n->D[l] = nz >> l;
        n->nv[l] = (long)n->W[l] * n->H[l] * n->D[l];
    }
    long off = 0;
    for (int l = 0; l < NL; ++l) {
        Layer& L = n->L[l];
        L.cin = CIN[l];
        L.cout = COUT[l];
        L.level = LEVEL[l];
        L.w_off = off;
        off += 27L * L.cin * L.cout;
        L.b_off = off;
        off += L.cout;
        L.kb_f = (27 * L.cin + 31) / 32;
        L.kb_b = (27 * L.cout + 31) / 32;
    }
    n->head_off = off;
    off += 17;
    n->nparam = off;
    n->capacity = capacity;
    hipError_t e = hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreate(&n->ev0);
    if (e == hipSuccess) e = hipEventCreate(&n->ev1);
    auto al = [&](void** p, size_t bytes) {
        if (e == hipSuccess) e = hipMalloc(p, bytes > 0 ? bytes : 16);
    };
    al((void**)&n->p, sizeof(float) * n->nparam);
    al((void**)&n->g, sizeof(float) * n->nparam);
    al((void**)&n->m1, sizeof(float) * n->nparam);
    al((void**)&n->m2, sizeof(float) * n->nparam);
    for (int l = 0; l < NL; ++l) {
        Layer& L = n->L[l];
        al((void**)&L.wf, 2ull * L.kb_f * 32 * L.cout);
        al((void**)&L.wb, 2ull * L.kb_b * 32 * L.cin);
        al((void**)&n->a[l], 2ull * n->nv[L.level] * L.cout);
        al((void**)&n->d[l], 2ull * n->nv[L.level] * L.cout);
    }
    al((void**)&n->x0, 2ull * n->nv[0] * 4);
    al((void**)&n->p1, 2ull * n->nv[1] * 16);
    al((void**)&n->p3, 2ull * n->nv[2] * 32);
    al((void**)&n->gc6, 2ull * n->nv[1] * 96);
    al((void**)&n->gc8, 2ull * n->nv[0] * 48);
    al((void**)&n->gp1, 2ull * n->nv[1] * 16);
    al((void**)&n->gp3, 2ull * n->nv[2] * 32);
    al((void**)&n->out, 4ull * n->nv[0]);
    al((void**)&n->feat, 4ull * 5 * n->nv[0]);
    al((void**)&n->red, 16);
    n->wpart_n = 0;
    for (int l = 0; l < NL; ++l) {
        const Layer& L = n->L[l];
        BrickPlan bp;
        if (brick_plan(n->ncu, n->D[L.level], n->H[L.level], n->W[L.level], L.cin, L.cout, &bp))
            n->wpart_n = std::max(n->wpart_n, (long)bp.ny * bp.nb * bp.per);
    }
    if (n->wpart_n > 0) al((void**)&n->wpart, sizeof(float) * n->wpart_n);
    al((void**)&n->ds_feat, 8ull * n->nv[0] * (capacity > 0 ? capacity : 1));
    al((void**)&n->ds_tgt, 4ull * n->nv[0] * (capacity > 0 ? capacity : 1));
    if (e != hipSuccess) {
        g_dn_err = std::string("denoiser allocation: ") + hipGetErrorString(e);
        tam_dn_destroy(n);
        return e == hipErrorOutOfMemory ? TAM_ERR_NOMEM : TAM_ERR_HIP;
    }
    // He initialisation (input layer: 4 real channels; the 12 padding
    // channels always see zeros), zero biases, zero head (output = input)
    std::vector<float> h((size_t)n->nparam, 0.f);
    std::mt19937_64 rng(seed);
    for (int l = 0; l < NL; ++l) {
        const Layer& L = n->L[l];
        const int fan = 27 * (l == 0 ? 4 : L.cin);
        std::normal_distribution<float> nd(0.f, std::sqrt(2.f / (float)fan));
        for (int t = 0; t < 27; ++t)
            for (int ci = 0; ci < L.cin; ++ci)
                for (int co = 0; co < L.cout; ++co)
                    h[(size_t)(L.w_off + ((long)t * L.cin + ci) * L.cout + co)] = (l == 0 && ci >= 4) ? 0.f : nd(rng);
    }
    e = hipMemcpy(n->p, h.data(), sizeof(float) * h.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(n->m1, 0, sizeof(float) * n->nparam);
    if (e == hipSuccess) e = hipMemset(n->m2, 0, sizeof(float) * n->nparam);
    if (e == hipSuccess) e = repack(n);
    if (e == hipSuccess) e = hipStreamSynchronize(n->stream);
    if (e != hipSuccess) {
        g_dn_err = std::string("denoiser init: ") + hipGetErrorString(e);
        tam_dn_destroy(n);
        return TAM_ERR_HIP;
    }
    *out = n;
    return TAM_OK;
}

void tam_dn_destroy(tam_dn* n)
{
    if (!n) return;
    DevScope ds(n->dev);
    if (n->stream) hipStreamSynchronize(n->stream);
    std::vector<void*> ptrs = {n->p, n->g, n->m1, n->m2, n->x0, n->p1, n->p3, n->gc6, n->gc8,
                               n->gp1, n->gp3, n->out, n->feat, n->red, n->ds_feat, n->ds_tgt, n->wpart};
    for (int l = 0; l < NL; ++l) {
        ptrs.push_back(n->L[l].wf);
        ptrs.push_back(n->L[l].wb);
        ptrs.push_back(n->a[l]);
        ptrs.push_back(n->d[l]);
    }
    for (void* q : ptrs)
        if (q) hipFree(q);
    if (n->ev0) hipEventDestroy(n->ev0);
    if (n->ev1) hipEventDestroy(n->ev1);
    if (n->stream) hipStreamDestroy(n->stream);
    delete n;
}

const char* tam_dn_last_error(const tam_dn* n) { return n ? n->err.c_str() : g_dn_err.c_str(); }

int64_t tam_dn_num_params(const tam_dn* n) { return n ? n->nparam : -1; }

int tam_dn_get_params(tam_dn* n, float* out)
{
    if (!n || !out) return TAM_ERR_ARG;
    DevScope ds(n->dev);
    DNCHK(n, hipMemcpyAsync(out, n->p, sizeof(float) * n->nparam, hipMemcpyDeviceToHost, n->stream));
    DNCHK(n, hipStreamSynchronize(n->stream));
    return TAM_OK;
}

int tam_dn_set_params(tam_dn* n, const float* in)
{
    if (!n || !in) return TAM_ERR_ARG;
    DevScope ds(n->dev);
    DNCHK(n, hipMemcpyAsync(n->p, in, sizeof(float) * n->nparam, hipMemcpyHostToDevice, n->stream));
    DNCHK(n, hipMemsetAsync(n->m1, 0, sizeof(float) * n->nparam, n->stream));
    DNCHK(n, hipMemsetAsync(n->m2, 0, sizeof(float) * n->nparam, n->stream));
    n->step = 0;
    DNCHK(n, repack(n));
    DNCHK(n, hipStreamSynchronize(n->stream));
    return TAM_OK;
}

int tam_dn_store(tam_dn* n, int32_t slot, const tam_ctx* lo, double npk_lo, const tam_ctx* hi, double npk_hi)
{
    if (!n || !lo || !hi) return TAM_ERR_ARG;
    if (slot < 0 || slot >= n->capacity) return dfail(n, TAM_ERR_ARG, "slot out of range");
    if (lo->p.nx != n->W[0] || lo->p.ny != n->H[0] || lo->p.nz != n->D[0] || hi->p.nx != n->W[0] ||
        hi->p.ny != n->H[0] || hi->p.nz != n->D[0] || lo->dev != n->dev || hi->dev != n->dev)
        return dfail(n, TAM_ERR_ARG, "contexts must match the network's grid and device");
    if (!(npk_lo > 0 && npk_hi > 0)) return dfail(n, TAM_ERR_ARG, "packet counts must be positive");
    DevScope ds(n->dev);
    const long nv = n->nv[0];
    const double vcm = lo->p.volume_voxel * 1e6;
    // the contexts' streams finish their transport before this stream reads
    DNCHK(n, hipStreamSynchronize(lo->stream));
    DNCHK(n, hipStreamSynchronize(hi->stream));
    hipLaunchKernelGGL(ctx_features_kernel, dim3(grid_of(nv)), dim3(256), 0, n->stream, lo->tally, lo->mut, lo->mat,
                       lo->mtab, nv, 1.0 / (npk_lo * vcm), n->feat);
    hipLaunchKernelGGL(store_slot_kernel, dim3(grid_of(nv)), dim3(256), 0, n->stream, n->feat, hi->tally,
                       1.0 / (npk_hi * vcm), nv, n->ds_feat + (long)slot * nv * 4, n->ds_tgt + (long)slot * nv);
    DNCHK(n, hipGetLastError());
    DNCHK(n, hipStreamSynchronize(n->stream));
    return TAM_OK;
}

int tam_dn_store_host(tam_dn* n, int32_t slot, const float* features, const float* target)
{
    if (!n || !features || !target) return TAM_ERR_ARG;
    if (slot < 0 || slot >= n->capacity) return dfail(n, TAM_ERR_ARG, "slot out of range");
    DevScope ds(n->dev);
    const long nv = n->nv[0];
    DNCHK(n, hipMemcpyAsync(n->feat, features, sizeof(float) * 4 * nv, hipMemcpyHostToDevice, n->stream));
    DNCHK(n, hipMemcpyAsync(n->feat + 4 * nv, target, sizeof(float) * nv, hipMemcpyHostToDevice, n->stream));
    hipLaunchKernelGGL(store_slot_kernel, dim3(grid_of(nv)), dim3(256), 0, n->stream, n->feat, (const double*)nullptr,
                       0.0, nv, n->ds_feat + (long)slot * nv * 4, n->ds_tgt + (long)slot * nv);
    DNCHK(n, hipGetLastError());
    DNCHK(n, hipStreamSynchronize(n->stream));
    return TAM_OK;
}

int tam_dn_train(tam_dn* n, int32_t nslots, int32_t steps, double lr, uint64_t seed, float* losses)
{
    if (!n) return TAM_ERR_ARG;
    if (nslots < 1 || nslots > n->capacity || steps < 0 || !(lr > 0))
        return dfail(n, TAM_ERR_ARG, "need 1 <= nslots <= capacity, steps >= 0, lr > 0");
    DevScope ds(n->dev);
    const long nv = n->nv[0];
    std::mt19937_64 rng(seed);
    std::vector<double> red((size_t)steps > 0 ? (size_t)steps * 2 : 2);
    double* dred = nullptr;
    DNCHK(n, hipMalloc((void**)&dred, sizeof(double) * 2 * (size_t)(steps > 0 ? steps : 1)));
    DNCHK(n, hipEventRecord(n->ev0, n->stream));
    hipError_t e = hipSuccess;
    for (int s = 0; s < steps && e == hipSuccess; ++s) {
        const int slot = (int)(rng() % (uint64_t)nslots);
        const float* tgt = n->ds_tgt + (long)slot * nv;
        const uint16_t* x0 = n->ds_feat + (long)slot * nv * 4;    // a slot holds the input's layout
        e = forward(n, x0, tgt);
        if (e == hipSuccess) e = hipMemcpyAsync(dred + 2 * s, n->red, 16, hipMemcpyDeviceToDevice, n->stream);
        if (e == hipSuccess) e = backward(n, x0, tgt);
        if (e == hipSuccess) e = adam(n, (float)lr);
    }
    if (e == hipSuccess) e = hipEventRecord(n->ev1, n->stream);
    if (e == hipSuccess && steps > 0)
        e = hipMemcpyAsync(red.data(), dred, sizeof(double) * 2 * steps, hipMemcpyDeviceToHost, n->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(n->stream);
    hipFree(dred);
    if (e != hipSuccess) return dfail(n, TAM_ERR_HIP, std::string("training: ") + hipGetErrorString(e));
    n->last_ms = ms_between(n);
    if (losses)
        for (int s = 0; s < steps; ++s) losses[s] = (float)(red[2 * (size_t)s] / (double)nv);
    return TAM_OK;
}

int tam_dn_eval(tam_dn* n, int32_t slot, double* l1_pred, double* l1_input)
{
    if (!n) return TAM_ERR_ARG;
    if (slot < 0 || slot >= n->capacity) return dfail(n, TAM_ERR_ARG, "slot out of range");
    DevScope ds(n->dev);
    const long nv = n->nv[0];
    const float* tgt = n->ds_tgt + (long)slot * nv;
    DNCHK(n, hipEventRecord(n->ev0, n->stream));
    DNCHK(n, forward(n, n->ds_feat + (long)slot * nv * 4, tgt));
    DNCHK(n, hipEventRecord(n->ev1, n->stream));
    double r[2];
    DNCHK(n, hipMemcpyAsync(r, n->red, 16, hipMemcpyDeviceToHost, n->stream));
    DNCHK(n, hipStreamSynchronize(n->stream));
    n->last_ms = ms_between(n);
    if (l1_pred) *l1_pred = r[0] / (double)nv;
    if (l1_input) *l1_input = r[1] / (double)nv;
    return TAM_OK;
}

int tam_dn_predict_slot(tam_dn* n, int32_t slot, float* pred, float* target, float* input)
{
    if (!n) return TAM_ERR_ARG;
    if (slot < 0 || slot >= n->capacity) return dfail(n, TAM_ERR_ARG, "slot out of range");
    DevScope ds(n->dev);
    const long nv = n->nv[0];
    DNCHK(n, forward(n, n->ds_feat + (long)slot * nv * 4, nullptr));
    if (pred) DNCHK(n, hipMemcpyAsync(pred, n->out, sizeof(float) * nv, hipMemcpyDeviceToHost, n->stream));
    if (target)
        DNCHK(n, hipMemcpyAsync(target, n->ds_tgt + (long)slot * nv, sizeof(float) * nv, hipMemcpyDeviceToHost,
                                n->stream));
    if (input) {
        std::vector<uint16_t> f((size_t)nv * 4);
        DNCHK(n, hipMemcpyAsync(f.data(), n->ds_feat + (long)slot * nv * 4, 8 * (size_t)nv, hipMemcpyDeviceToHost,
                                n->stream));
        DNCHK(n, hipStreamSynchronize(n->stream));
        for (long m = 0; m < nv; ++m) {
            const uint32_t u = (uint32_t)f[(size_t)m * 4] << 16;
            float v;
            std::memcpy(&v, &u, 4);
            input[m] = v;
        }
    }
    DNCHK(n, hipStreamSynchronize(n->stream));
    return TAM_OK;
}

int tam_dn_forward_host(tam_dn* n, const float* features, float* out)
{
    if (!n || !features || !out) return TAM_ERR_ARG;
    DevScope ds(n->dev);
    const long nv = n->nv[0];
    DNCHK(n, hipMemcpyAsync(n->feat, features, sizeof(float) * 4 * nv, hipMemcpyHostToDevice, n->stream));
    hipLaunchKernelGGL(pack_input_kernel, dim3(grid_of(nv)), dim3(256), 0, n->stream, n->feat, nv, n->x0);
    DNCHK(n, hipEventRecord(n->ev0, n->stream));
    DNCHK(n, forward(n, n->x0, nullptr));
    DNCHK(n, hipEventRecord(n->ev1, n->stream));
    DNCHK(n, hipMemcpyAsync(out, n->out, sizeof(float) * nv, hipMemcpyDeviceToHost, n->stream));
    DNCHK(n, hipStreamSynchronize(n->stream));
    n->last_ms = ms_between(n);
    return TAM_OK;
}

int tam_dn_gradients_host(tam_dn* n, const float* features, const float* target, float* grads, double* loss)
{
    if (!n || !features || !target || !grads) return TAM_ERR_ARG;
    if (n->capacity < 1) return dfail(n, TAM_ERR_ARG, "needs one dataset slot");
    DevScope ds(n->dev);
    const long nv = n->nv[0];
    const int rc = tam_dn_store_host(n, 0, features, target);
    if (rc != TAM_OK) return rc;
    const float* tgt = n->ds_tgt;
    DNCHK(n, forward(n, n->ds_feat, tgt));
    DNCHK(n, backward(n, n->ds_feat, tgt));
    double r[2];
    DNCHK(n, hipMemcpyAsync(r, n->red, 16, hipMemcpyDeviceToHost, n->stream));
    DNCHK(n, hipMemcpyAsync(grads, n->g, sizeof(float) * n->nparam, hipMemcpyDeviceToHost, n->stream));
    DNCHK(n, hipStreamSynchronize(n->stream));
    if (loss) *loss = r[0] / (double)nv;
    return TAM_OK;
}

int tam_dn_apply(tam_dn* n, tam_ctx* c, double npk)
{
    if (!n || !c) return TAM_ERR_ARG;
    if (c->p.nx != n->W[0] || c->p.ny != n->H[0] || c->p.nz != n->D[0] || c->dev != n->dev)
        return dfail(n, TAM_ERR_ARG, "the context must match the network's grid and device");
    if (!(npk > 0)) return dfail(n, TAM_ERR_ARG, "packet count must be positive");
    DevScope ds(n->dev);
    const long nv = n->nv[0];
    const double vcm = c->p.volume_voxel * 1e6;
    DNCHK(n, hipStreamSynchronize(c->stream));
    DNCHK(n, hipEventRecord(n->ev0, n->stream));
    hipLaunchKernelGGL(ctx_input_kernel, dim3(grid_of(nv)), dim3(256), 0, n->stream, c->tally, c->mut, c->mat,
                       c->mtab, nv, 1.0 / (npk * vcm), n->x0);
    DNCHK(n, forward(n, n->x0, nullptr, c, npk * vcm));
    DNCHK(n, hipEventRecord(n->ev1, n->stream));
    DNCHK(n, hipStreamSynchronize(n->stream));
    n->last_ms = ms_between(n);
    return TAM_OK;
}

double tam_dn_last_ms(const tam_dn* n) { return n ? (double)n->last_ms : 0.0; }

}  // extern "C"
