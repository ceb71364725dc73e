// Learned warm start of the multigrid solve: a 3D U-Net on gfx950 matrix
// cores.  Activations and weights are BF16, channels last
// ([batch][z][y][x][channel]); every 3^3 convolution is an implicit GEMM on
// v_mfma_f32_16x16x32_bf16 with FP32 accumulation:
//   forward      out[v][co] = b[co] + sum_{t, ci} in[v + off_t][ci] W[t][ci][co]
//                (rows = 16 voxels along x, columns = 16 output channels,
//                K = 27 taps x input channels in chunks of 8);
//   input grad   the same kernel on the output gradient with the taps mirrored
//                and W transposed;
//   weight grad  dW[t][ci][co] = sum_v in[v + off_t][ci] dout[v][co]
//                (rows = output channels, columns = input channels, K =
//                voxels of a 16x4x4 brick staged in LDS), per-chunk FP32
//                partials summed in a fixed order.
// The grid is periodic (the multigrid problem is), so every convolution wraps.
// A decoder convolution reads its skip input at full resolution and the
// coarser level's features through a nearest-neighbour upsampling on read,
// so the concatenation is never stored.  The reference has no counterpart:
// it seeds nothing (src/multigrid.jl:722-752 starts every level from zero).
#include <math.h>
#include <string.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "kernels.hpp"

namespace baorec {
namespace unet {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
// round to nearest even, the conversion instruction (the bit operations it
// replaces were a fourth of a convolution's vector instructions)
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

__device__ __forceinline__ bf16x8 load8(const uint16_t *p) {
    const uint4 q = *reinterpret_cast<const uint4 *>(p);
    return __builtin_bit_cast(bf16x8, q);
}

// zeroes the gradients h of outputs y of a ReLU that are not positive
template <int N>
__device__ __forceinline__ void relu_mask(uint16_t *h, const uint16_t *y) {
#pragma unroll
    for (int j = 0; j < N; j++)
        if (!(bf2f(y[j]) > 0.f)) h[j] = 0;
}

// ------------------------------------------------------------ convolution

// Tiling of k_conv: a workgroup of four waves computes 16 x MB x ZW voxels
// (wave: one z plane, MB rows of 16 voxels) times 16 NB CW output channels
// (CW waves share a plane), the output channels split over NSPLIT workgroups.
// An operand read from LDS (1 KB) feeds NB products, a weight read (1 KB from
// L1) MB of them, so MB and NB are as large as LDS (18 (MB + 2) (ZW + 2)
// voxels) and registers allow with at least two workgroups per CU where the
// channels permit; the coarse levels' many channels split over workgroups
// instead, since their grids are few voxels.
//
// The whole tile with its halo stands in LDS before the products start (each
// input voxel is an operand 27 times; read from memory each time, L1 delivered
// 64 bytes per cycle and CU and bound the kernel).  Weights are the products'
// first operand and voxels their second, so that a lane ends with four
// channels of one voxel and stores 8 bytes.  Products per output run in
// ascending K, one chain.
//
// Measured on a batch of four 128^3 grids (before: operands from L1): 16 -> 16
// channels 156 us (436; 537 MB, 115 us at the copy rate), with a ReLU mask 199,
// 48 -> 16 532 (1357), 16 -> 48 353 (828; 1.07 GB, 225 us), 96 -> 32 at 64^3
// 245 (541).  The 16-channel outputs are bound by LDS: every product needs
// 1 KB at 128 bytes per cycle and CU, 104 us for 16 -> 16, 305 us for 48 -> 16.
template <int CIN, int CO>
struct ConvTile {
    static constexpr int MB = CIN <= 16 ? 8 : CIN <= 96 ? 4 : 2;
    static constexpr int ZW = CIN == 64 || CIN >= 128 ? 2 : 4, CW = 4 / ZW;
    static constexpr int NBW = CO / 16 / CW;   // blocks of 16 output channels per wave, over all splits
    static constexpr int NB = CIN == 128 ? 1 : NBW % 3 == 0 ? 3 : NBW % 2 == 0 ? 2 : 1;
    static constexpr int NSPLIT = NBW / NB;
    // uint16 per voxel in LDS.  An operand read (16 voxels at this stride, lane
    // groups 1 and 3 a piece of 16 bytes further than 0 and 2) is free of bank
    // conflicts at 2 mod 4 pieces, or at 4 mod 8 with piece p of voxel hx stored
    // at p ^ swz(hx); 128 channels take 17, for two workgroups per CU.
    static constexpr bool SWZ = CIN % 64 == 32;
    static constexpr int VS = CIN == 128 ? CIN + 8 : CIN % 64 == 0 ? CIN + 16 : CIN;
    static __device__ __forceinline__ int swz(int hx) { return SWZ ? (hx >> 1) & 2 : 0; }
    static constexpr int HY = MB + 2, HZ = ZW + 2;
    static constexpr int LDS = 18 * HY * HZ * VS;
    // the layers' input gradients that may carry a ReLU mask
    static constexpr bool maskable(bool relu) { return !relu && CIN == CO; }
    static constexpr int FIT = 160 * 1024 / (2 * LDS);   // workgroups per CU
    static constexpr int WGS = MB * NB < 16 && FIT >= 3 ? (FIT >= 4 ? 4 : 3) : FIT >= 2 ? 2 : 1;
};

template <int C1, int C2, int CO, bool RELU, bool UP2>
__global__ void __launch_bounds__(256, (ConvTile<C1 + C2, CO>::WGS)) k_conv(ConvArgs a) {
    constexpr int CIN = C1 + C2;
    using T = ConvTile<CIN, CO>;
    constexpr int KB = (27 * CIN + 31) / 32;
    constexpr bool MASKED = T::maskable(RELU);
    constexpr int NBT = CO / 16, NB = T::NB, MB = T::MB, HY = T::HY, HZ = T::HZ, VS = T::VS;
    static_assert(C1 % 8 == 0 && C2 % 8 == 0 && CO % 16 == 0 && NB * T::CW * T::NSPLIT == NBT, "channel blocks");
    __shared__ __align__(16) uint16_t tile[T::LDS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int nx = 1 << a.lx, ny = 1 << a.ly, nz = 1 << a.lz;
    const int x0 = blockIdx.x * 16, y0 = blockIdx.y * MB;
    const int split = blockIdx.z % T::NSPLIT, zb = blockIdx.z / T::NSPLIT;
    const int lzt = a.lz > (T::ZW == 4 ? 2 : 1) ? a.lz - (T::ZW == 4 ? 2 : 1) : 0;   // log2 of the z tiles
    const int z0 = (zb & ((1 << lzt) - 1)) * T::ZW;
    const uint32_t b = zb >> lzt;
    const int zw = wave % T::ZW, nb0 = (split * T::CW + wave / T::ZW) * NB;   // the wave's plane and first block
    // weights of chunk kb
    const uint16_t *wl = a.w + (((uint32_t)nb0 * 4 + g) * 16 + r16) * 8;
    auto load_w = [&](int kb, bf16x8 *q) {
#pragma unroll
        for (int nb = 0; nb < NB; nb++) q[nb] = load8(wl + (uint32_t)(kb * NBT + nb) * 512);
    };
    // rings of operand sets, indexed statically.  Weights beyond half of L1
    // come from L2 and are asked for about 700 cycles of products ahead.
    constexpr int RW = KB * NBT > 16 ? (MB * NB <= 8 ? 8 : MB * NB <= 16 ? 4 : 2) : MB * NB >= 16 ? 2 : 4;
    constexpr int RA = MB >= 4 ? 2 : 4;
    bf16x8 wq[RW][NB], aq[RA][MB];
#pragma unroll
    for (int i = 0; i < RW - 1; i++) load_w(i, wq[i]);
    // the tile and its one-cell periodic halo: channels [coff, coff + C) of it
    // from src, a grid of sides halved l times; a thread moves one 16-byte piece
    // of every (256 / S)-th voxel, eight loads in flight
    auto fill = [&](auto C_, int coff, const uint16_t *src, int l) {
        constexpr int C = decltype(C_)::value, S = C / 8, STEP = 256 / S, NV = 18 * HY * HZ;
        constexpr int IT = (NV + STEP - 1) / STEP, U = 8;
        const int slot = tid % S, v0 = tid / S;
        int hx = v0 % 18, row = v0 / 18;
        uint16_t *dst = tile + v0 * VS;
#pragma unroll
        for (int i0 = 0; i0 < IT; i0 += U) {
            f32x4 q[U];
            int off[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int hz = row / HY, hy = row - hz * HY;
                const uint32_t xs = (uint32_t)((x0 - 1 + hx) & (nx - 1)) >> l, ys = (uint32_t)((y0 - 1 + hy) & (ny - 1)) >> l;
                const uint32_t zs = (uint32_t)((z0 - 1 + hz) & (nz - 1)) >> l;
                const uint32_t zy = (((b << (a.lz - l)) + zs) << (a.ly - l)) + ys;
                off[u] = (coff / 8 + slot ^ T::swz(hx)) * 8;
                if (i0 + u < IT && v0 + (i0 + u) * STEP < NV)
                    q[u] = *reinterpret_cast<const f32x4 *>(src + ((zy << (a.lx - l)) + xs) * C + slot * 8);
                hx += STEP % 18;
                row += STEP / 18;
                if (STEP % 18 && hx >= 18) {
                    hx -= 18;
                    row++;
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (i0 + u < IT && v0 + (i0 + u) * STEP < NV)
                    *reinterpret_cast<f32x4 *>(dst + (i0 + u) * STEP * VS + off[u]) = q[u];
        }
    };
    fill(std::integral_constant<int, C1>{}, 0, a.in1, 0);
    if constexpr (C2 > 0) fill(std::integral_constant<int, C2>{}, C1, a.in2, UP2 ? 1 : 0);
    __syncthreads();
    const int x = x0 + r16, z = z0 + zw;   // the lane's voxels: y0 + m
    const uint32_t vox0 = (((((b << a.lz) + z) << a.ly) + y0) << a.lx) + x;   // (the launcher checks the sizes)
    uint2 mk[MB][NB];   // in flight during the products
    if (MASKED && a.mask)
#pragma unroll
        for (int m = 0; m < MB; m++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++) {
                mk[m][nb] = make_uint2(0u, 0u);
                if (x < nx && y0 + m < ny && z < nz)
                    mk[m][nb] = *reinterpret_cast<const uint2 *>(a.mask + (size_t)(vox0 + m * nx) * CO +
                                                                 (nb0 + nb) * 16 + 4 * g);
            }
    f32x4 acc[MB][NB];
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++) acc[m][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    // inputs of chunk kb: lane group g holds channels ci .. ci + 7 of tap t
    const uint16_t *al[3];
#pragma unroll
    for (int dx = 0; dx < 3; dx++)
        al[dx] = tile + (zw * HY * 18 + r16) * VS + (CIN % 16 == 0 ? (g ^ T::swz(r16 + dx)) * 8 : 0);
    const int m1 = -(g & 1), m2 = -(g >> 1);
    auto load_a = [&](int kb, bf16x8 *q) {
        auto off = [&](int gg) {   // from al
            const int kc = kb * 32 + gg * 8;
            const int t = kc / CIN, ci = kc - t * CIN;
            const int tt = t > 26 ? 26 : t;   // padding columns of K: their weights are zero
            return ((tt / 9 * HY + tt / 3 % 3) * 18 + tt % 3) * VS + ci - (CIN % 16 == 0 ? gg * 8 : 0);
        };
        const int t0 = kb * 32 / CIN;
        const uint16_t *p = al[t0 > 26 ? 2 : t0 % 3] + off(0);
        // the groups' taps differ where 32 is not within one tap's channels
        if (CIN % 32 != 0) p += m2 & (off(2) - off(0));
        if (CIN % 16 != 0) p += (m1 & ~m2 & (off(1) - off(0))) + (m1 & m2 & (off(3) - off(2)));
#pragma unroll
        for (int m = 0; m < MB; m++) q[m] = *reinterpret_cast<const bf16x8 *>(p + m * 18 * VS);
    };
#pragma unroll
    for (int i = 0; i < RA - 1; i++) load_a(i, aq[i]);
#pragma unroll
    for (int kb = 0; kb < KB; kb++) {
        if (kb + RW - 1 < KB) load_w(kb + RW - 1, wq[(kb + RW - 1) % RW]);
        if (kb + RA - 1 < KB) load_a(kb + RA - 1, aq[(kb + RA - 1) % RA]);
#pragma unroll
        for (int m = 0; m < MB; m++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
                acc[m][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wq[kb % RW][nb], aq[kb % RA][m], acc[m][nb], 0, 0, 0);
    }
    // lane holds channels 4g .. 4g+3 of voxel r16
    if (x >= nx || z >= nz) return;
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        const int co = (nb0 + nb) * 16 + 4 * g;
        f32x4 bias = f32x4{0.f, 0.f, 0.f, 0.f};
        if (a.bias)
#pragma unroll
            for (int r = 0; r < 4; r++) bias[r] = a.bias[co + r];
        // channels [csplit, CO) go to out2
        const bool second = !RELU && (nb0 + nb) * 16 >= a.csplit;
        const int stride = RELU ? CO : second ? CO - a.csplit : a.csplit;
        uint16_t *dst = (second ? a.out2 - a.csplit : a.out) + ((size_t)vox0 * stride + co);
#pragma unroll
        for (int m = 0; m < MB; m++, dst += (size_t)nx * stride) {
            if (y0 + m >= ny) break;
            uint16_t h[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float v = acc[m][nb][r] + bias[r];
                if (RELU) v = fmaxf(v, 0.f);
                h[r] = f2bf(v);
            }
            if (MASKED && a.mask) relu_mask<4>(h, reinterpret_cast<const uint16_t *>(&mk[m][nb]));
            *reinterpret_cast<uint2 *>(dst) = make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
        }
    }
}

// Weight gradient.  Workgroup: 16 input channels (block blockIdx.y / NBO), 16 NB
// output channels (block blockIdx.y % NBO), all 27 taps, bricks
// [chunk * per, (chunk + 1) * per) of 16 x 4 x 4 voxels.  A = dout^T (rows:
// output channels, K: the brick's voxels in x-fastest order, 32 per product),
// B = the input at the tap's offset (columns: input channels).  Both stand in
// LDS channels last, as in memory, and reach the matrix cores through the
// transposing LDS read (16 lanes fetch 4 voxels x 16 channels and each gets
// one channel's 4 voxels), so a product's operands cost 64-bit reads and no
// element moves.  Wave w owns the 9 taps with dy = w - 1: an input row pair
// read once (10 voxels per lane: the three dx are register shifts) feeds three
// dx times the up to three dz whose voxels lie in the brick; dout of the whole
// brick stays in registers.  Every tap's products run in ascending voxel
// order, one accumulator chain per chunk.  The next brick's global loads are
// in flight during the products; with one workgroup per chunk (a CU then has
// only this one) LDS is double buffered.
//
// LDS reads are free of bank conflicts: an input row has 128 spare bytes after
// every 8 voxels, so that the two 8-voxel halves a read touches lie in
// different halves of the banks, and dout's voxel 4-groups change places in
// every second 8-group.
//
// Measured on a batch of four 128^3 grids: 16 -> 16 channels 226 us (537 MB of
// inputs, 115 us at the copy rate; with element-wise LDS reads 1337), 48 -> 16
// 511 us (2517), 96 -> 32 at 64^3 269 us (1187).  With one workgroup of three
// waves per CU the finest layers are bound by the brick's load, store and
// barrier not fully hidden behind its 72 products per wave; the coarse ones by
// the partial sums of their chunks (up to 340 MB).
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint2 lds_read_tr(const uint16_t *p) {
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4 *)(__attribute__((address_space(3))) void *)p);
    return __builtin_bit_cast(uint2, v);
}
constexpr int kWgThreads = 192, kWgRow = 448;   // threads; uint16 per LDS row of 18 voxels (and 2 never used)
__host__ __device__ constexpr int wgrad_nb(int co) { return co >= 32 ? 2 : 1; }

template <int C1, int C2, int CO, bool UP2>
__global__ void __launch_bounds__(kWgThreads, 1) k_conv_wgrad(WgradArgs a) {
    constexpr int CIN = C1 + C2;
    constexpr int NB = wgrad_nb(CO), NBO = CO / (16 * NB);
    constexpr int BUFS = ((CIN + 15) / 16) * NBO == 1 ? 2 : 1;
    constexpr int NIN = 7, NDO = (512 * NB + kWgThreads - 1) / kWgThreads;   // 16-byte loads per thread
    __shared__ __align__(16) uint16_t sIn[BUFS][36 * kWgRow];
    __shared__ __align__(16) uint16_t sDo[BUFS][NB * 4096];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, g = lane >> 4;
    const int cib = blockIdx.y / NBO, cob = blockIdx.y % NBO;
    const int nx = 1 << a.lx, ny = 1 << a.ly, nz = 1 << a.lz;
    // log2 of the bricks along each axis
    const int lbx = a.lx > 4 ? a.lx - 4 : 0, lby = a.ly > 2 ? a.ly - 2 : 0, lbz = a.lz > 2 ? a.lz - 2 : 0;
    const int nbricks = a.batch << (lbx + lby + lbz);
    f32x4 acc[NB][3][3];   // [][dz][dx]
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
        for (int i = 0; i < 9; i++) acc[n][i / 3][i % 3] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int beg = blockIdx.x * (int)a.per;
    const int end = nbricks - beg > a.per ? beg + (int)a.per : nbricks;

    // this thread's 16-byte pieces of a brick: half = 8 channels of voxel v of
    // the input with its one-cell halo (18 x 6 x 6), and of dout (16 x 4 x 4)
    const int half = tid & 1;
    const bool skip = CIN < 16 && half == 1;   // 8 input channels: the rest are zero
    const int c = cib * 16 + half * 8;
    uint4 rin[NIN], rdo[NDO];
    // voxel index on the grid of sides halved l times
    auto vox = [&](uint32_t b, uint32_t z, uint32_t y, uint32_t x, int l) {
        const uint32_t zy = (((b << (a.lz - l)) + z) << (a.ly - l)) + y;
        return (zy << (a.lx - l)) + x;
    };
    auto load = [&](int br) {
        const int x0 = (br & ((1 << lbx) - 1)) * 16, y0 = ((br >> lbx) & ((1 << lby) - 1)) * 4;
        const int z0 = ((br >> (lbx + lby)) & ((1 << lbz) - 1)) * 4;
        const uint32_t b = (uint32_t)br >> (lbx + lby + lbz);
#pragma unroll
        for (int u = 0; u < NIN; u++) {
            const int v = (tid >> 1) + (kWgThreads / 2) * u;
            rin[u] = make_uint4(0u, 0u, 0u, 0u);
            if (v >= 648 || skip) continue;
            const int hx = v % 18, hy = (v / 18) % 6, hz = v / 108;
            const int xs = (x0 - 1 + hx) & (nx - 1), ys = (y0 - 1 + hy) & (ny - 1), zs = (z0 - 1 + hz) & (nz - 1);
            const uint16_t *src;
            if (C2 == 0 || cib * 16 < C1) {
                src = a.in1 + vox(b, zs, ys, xs, 0) * C1 + c;
            } else if (UP2) {
                src = a.in2 + vox(b, zs >> 1, ys >> 1, xs >> 1, 1) * C2 + (c - C1);
            } else {
                src = a.in2 + vox(b, zs, ys, xs, 0) * C2 + (c - C1);
            }
            rin[u] = *reinterpret_cast<const uint4 *>(src);
        }
#pragma unroll
        for (int u = 0; u < NDO; u++) {
            const int i = tid + kWgThreads * u, h = i % (2 * NB), v = i / (2 * NB);
            rdo[u] = make_uint4(0u, 0u, 0u, 0u);
            const int x = x0 + (v & 15), y = y0 + ((v >> 4) & 3), z = z0 + (v >> 6);
            if (v < 256 && x < nx && y < ny && z < nz)
                rdo[u] = *reinterpret_cast<const uint4 *>(a.dout + vox(b, z, y, x, 0) * CO +
                                                          cob * 16 * NB + h * 8);
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int u = 0; u < NIN; u++) {
            const int v = (tid >> 1) + (kWgThreads / 2) * u;
            const int hx = v % 18, row = v / 18;   // row = hz * 6 + hy
            if (v < 648)
                *reinterpret_cast<uint4 *>(&sIn[buf][row * kWgRow + hx * 16 + (hx >> 3) * 64 + half * 8]) = rin[u];
        }
#pragma unroll
        for (int u = 0; u < NDO; u++) {
            const int i = tid + kWgThreads * u, h = i % (2 * NB), v = i / (2 * NB);
            if (v < 256)
                *reinterpret_cast<uint4 *>(
                    &sDo[buf][(h >> 1) * 4096 + (v ^ ((v >> 1) & 4)) * 16 + (h & 1) * 8]) = rdo[u];
        }
    };
    auto compute = [&](int buf) {
        uint4 av[NB][8];
        const uint16_t *d0 = &sDo[buf][g * 128 + (g & 1) * 64 + r16 * 4];
        const uint16_t *d1 = &sDo[buf][g * 128 + 64 - (g & 1) * 64 + r16 * 4];
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int kb = 0; kb < 8; kb++) {
                const uint2 lo = lds_read_tr(d0 + n * 4096 + kb * 512), hi = lds_read_tr(d1 + n * 4096 + kb * 512);
                av[n][kb] = make_uint4(lo.x, lo.y, hi.x, hi.y);
            }
        const uint16_t *in0 = &sIn[buf][((g >> 1) + wave) * kWgRow + (g & 1) * 192 + r16 * 4];
#pragma unroll
        for (int zi = 0; zi < 6; zi++)
#pragma unroll
            for (int yp = 0; yp < 2; yp++) {
                const uint16_t *row = in0 + (zi * 6 + 2 * yp) * kWgRow;
                const uint2 p = lds_read_tr(row), q = lds_read_tr(row + 64), r = lds_read_tr(row + 192);
                const uint4 bv[3] = {make_uint4(p.x, p.y, q.x, q.y),
                                     make_uint4(__builtin_amdgcn_alignbit(p.y, p.x, 16),
                                                __builtin_amdgcn_alignbit(q.x, p.y, 16),
                                                __builtin_amdgcn_alignbit(q.y, q.x, 16),
                                                __builtin_amdgcn_alignbit(r.x, q.y, 16)),
                                     make_uint4(p.y, q.x, q.y, r.x)};
#pragma unroll
                for (int dz = 0; dz < 3; dz++) {
                    const int zk = zi - dz;
                    if (zk < 0 || zk > 3) continue;
#pragma unroll
                    for (int n = 0; n < NB; n++)
#pragma unroll
                        for (int dx = 0; dx < 3; dx++)
                            acc[n][dz][dx] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                __builtin_bit_cast(bf16x8, av[n][2 * zk + yp]), __builtin_bit_cast(bf16x8, bv[dx]),
                                acc[n][dz][dx], 0, 0, 0);
                }
            }
    };
    load(beg);
    store(0);
    __syncthreads();
    int buf = 0;
    for (int br = beg; br < end; br++) {
        const bool more = br + 1 < end;
        if (more) load(br + 1);
        compute(buf);
        if (BUFS == 2) buf ^= 1;
        else __syncthreads();
        if (more) store(buf);
        __syncthreads();
    }
    // D[row = output channel 4g + r][column = input channel r16]
    const int ci = cib * 16 + r16;
    if (ci >= CIN) return;
    float *part = a.part + (size_t)blockIdx.x * 27 * CIN * CO;
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
        for (int dz = 0; dz < 3; dz++)
#pragma unroll
            for (int dx = 0; dx < 3; dx++) {
                const int t = dz * 9 + wave * 3 + dx;
                *reinterpret_cast<f32x4 *>(part + ((size_t)t * CIN + ci) * CO + (cob * NB + n) * 16 + 4 * g) =
                    acc[n][dz][dx];
            }
}

// out[i] = sum over chunks c of part[c][i], c in order
__global__ void k_sum_chunks(const float *__restrict__ part, int nch, int64_t n, float *__restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        float s = 0.f;
        int c = 0;
        for (; c + 16 <= nch; c += 16) {   // 16 loads in flight, added in order
            float v[16];
#pragma unroll
            for (int j = 0; j < 16; j++) v[j] = part[(size_t)(c + j) * n + i];
#pragma unroll
            for (int j = 0; j < 16; j++) s += v[j];
        }
        for (; c < nch; c++) s += part[(size_t)c * n + i];
        out[i] = s;
    }
}

// ------------------------------------------------------------ packing

// Master FP32 weights W[t][ci][co] -> the B operand of k_conv:
// [kb][nb][g][n][8] with k = kb*32 + g*8 + j = t*CIN + ci, co = nb*16 + n.
// transposed != 0 packs the input-gradient convolution instead: its K runs
// over (mirrored tap 26 - t, fwd output channel), its columns over the fwd
// input channels.
__global__ void k_pack(const float *__restrict__ w, int cin, int co, int transposed, uint16_t *__restrict__ out) {
    const int kin = transposed ? co : cin;     // K channels of the packed conv
    const int nout = transposed ? cin : co;    // its output channels
    const int KB = (27 * kin + 31) / 32, NB = nout / 16;
    const int64_t total = (int64_t)KB * NB * 4 * 16 * 8;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(e & 7);
        int64_t q = e >> 3;
        const int n = (int)(q & 15);
        q >>= 4;
        const int gg = (int)(q & 3);
        q >>= 2;
        const int nb = (int)(q % NB);
        const int kb = (int)(q / NB);
        const int k = kb * 32 + gg * 8 + j;
        const int t = k / kin, c = k - t * kin;
        const int col = nb * 16 + n;
        float v = 0.f;
        if (t < 27) v = transposed ? w[((size_t)(26 - t) * cin + col) * co + c] : w[((size_t)t * cin + c) * co + col];
        out[e] = f2bf(v);
    }
}

// ------------------------------------------------------------ elementwise

// The pooling and upsampling kernels below take a thread per voxel and 8
// channels (16-byte accesses; c = 1 << lc channels) and are bound by their
// traffic.

// 2x2x2 average pooling of a [b][z][y][x][c] tensor: nout voxels and 8-channel
// groups of the result
__global__ void k_pool(const uint16_t *__restrict__ in, uint16_t *__restrict__ out, int lx, int ly, int lc,
                       int64_t nout) {
    const int lg = lc - 3;   // log2 of the channel groups
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nout; i += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(i & ((1 << lg) - 1));
        const int64_t v = i >> lg;
        const int64_t x = v & ((1 << (lx - 1)) - 1), y = (v >> (lx - 1)) & ((1 << (ly - 1)) - 1), bz = v >> (lx + ly - 2);
        float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < 8; d++) {
            // batch and z together: the fine z of item b is 2 (b cz + z) + dz
            const int64_t f = ((((2 * bz + (d >> 2)) << ly) + 2 * y + ((d >> 1) & 1)) << lx) + 2 * x + (d & 1);
            const uint4 q = *reinterpret_cast<const uint4 *>(in + (f << lc) + c * 8);
            const uint16_t *h = reinterpret_cast<const uint16_t *>(&q);
#pragma unroll
            for (int j = 0; j < 8; j++) s[j] += bf2f(h[j]);
        }
        uint4 o;
        uint16_t *oh = reinterpret_cast<uint16_t *>(&o);
#pragma unroll
        for (int j = 0; j < 8; j++) oh[j] = f2bf(s[j] * 0.125f);
        *reinterpret_cast<uint4 *>(out + i * 8) = o;
    }
}

// dfine += dcoarse / 8 at the parent (the adjoint of k_pool), then zero where
// the fine output y is not positive: dfine's last term, so masked here
__global__ void k_pool_bwd(const uint16_t *__restrict__ dc, const uint16_t *__restrict__ y, uint16_t *__restrict__ df,
                           int lx, int ly, int lc, int64_t nfine) {
    const int lg = lc - 3;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nfine; i += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(i & ((1 << lg) - 1));
        const int64_t v = i >> lg;
        const int64_t vx = v & ((1 << lx) - 1), vy = (v >> lx) & ((1 << ly) - 1), bz = v >> (lx + ly);
        const int64_t p = ((((bz >> 1) << (ly - 1)) + (vy >> 1)) << (lx - 1)) + (vx >> 1);
        const uint4 qc = *reinterpret_cast<const uint4 *>(dc + (p << lc) + c * 8);
        const uint4 qy = *reinterpret_cast<const uint4 *>(y + i * 8);
        uint4 qf = *reinterpret_cast<const uint4 *>(df + i * 8);
        const uint16_t *hc = reinterpret_cast<const uint16_t *>(&qc);
        uint16_t *hf = reinterpret_cast<uint16_t *>(&qf);
#pragma unroll
        for (int j = 0; j < 8; j++) hf[j] = f2bf(bf2f(hf[j]) + bf2f(hc[j]) * 0.125f);
        relu_mask<8>(hf, reinterpret_cast<const uint16_t *>(&qy));
        *reinterpret_cast<uint4 *>(df + i * 8) = qf;
    }
}

// Gradient of a decoder's upsampled input (full resolution, C channels):
// dcoarse = its sum over the 8 children of each coarse cell (overwrites), zero
// where the coarse output y is not positive.  C / 8 a power of two.
__global__ void k_upsample_bwd(const uint16_t *__restrict__ dup, const uint16_t *__restrict__ y,
                               uint16_t *__restrict__ dcoarse, int lx, int ly, int lc, int64_t ncoarse) {
    const int lg = lc - 3;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < ncoarse; i += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(i & ((1 << lg) - 1));
        const int64_t v = i >> lg;
        const int64_t x = v & ((1 << (lx - 1)) - 1), vy = (v >> (lx - 1)) & ((1 << (ly - 1)) - 1);
        const int64_t bz = v >> (lx + ly - 2);
        float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < 8; d++) {
            const int64_t f = ((((2 * bz + (d >> 2)) << ly) + 2 * vy + ((d >> 1) & 1)) << lx) + 2 * x + (d & 1);
            const uint4 q = *reinterpret_cast<const uint4 *>(dup + (f << lc) + c * 8);
            const uint16_t *h = reinterpret_cast<const uint16_t *>(&q);
#pragma unroll
            for (int j = 0; j < 8; j++) s[j] += bf2f(h[j]);
        }
        const uint4 qy = *reinterpret_cast<const uint4 *>(y + i * 8);
        uint4 o;
        uint16_t *oh = reinterpret_cast<uint16_t *>(&o);
#pragma unroll
        for (int j = 0; j < 8; j++) oh[j] = f2bf(s[j]);
        relu_mask<8>(oh, reinterpret_cast<const uint16_t *>(&qy));
        *reinterpret_cast<uint4 *>(dcoarse + i * 8) = o;
    }
}

// Output layer: out[v] = b + sum_c w[c] x[v][c] (16 channels, FP32 out)
__global__ void k_head(const uint16_t *__restrict__ x, const float *__restrict__ w, const float *__restrict__ b,
                       float *__restrict__ out, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const uint4 q0 = *reinterpret_cast<const uint4 *>(x + i * 16);
        const uint4 q1 = *reinterpret_cast<const uint4 *>(x + i * 16 + 8);
        const uint16_t *h0 = reinterpret_cast<const uint16_t *>(&q0);
        const uint16_t *h1 = reinterpret_cast<const uint16_t *>(&q1);
        float s = b[0];
        for (int c = 0; c < 8; c++) s += w[c] * bf2f(h0[c]);
        for (int c = 0; c < 8; c++) s += w[8 + c] * bf2f(h1[c]);
        out[i] = s;
    }
}
// dx[v][c] = w[c] dout[v], zero where x[v][c] is not positive (x a ReLU's
// output); per-block partials of dw[c] = sum_v x[v][c] dout[v]
// and db = sum_v dout[v] (17 values per block, summed later by k_sum_rows).
// Bound by its traffic (32 B read and written and 4 B read per voxel): a
// voxel's 16 channels move as two 16-byte accesses each way.
__global__ void __launch_bounds__(256) k_head_bwd(const uint16_t *__restrict__ x, const float *__restrict__ w,
                                                  const float *__restrict__ dout, uint16_t *__restrict__ dx,
                                                  float *__restrict__ part, int64_t n) {
    __shared__ float red[17][4];
    float acc[17], wr[16];
#pragma unroll
    for (int c = 0; c < 17; c++) acc[c] = 0.f;
#pragma unroll
    for (int c = 0; c < 16; c++) wr[c] = w[c];
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float d = dout[i];
        uint4 q[2], o[2];
        q[0] = *reinterpret_cast<const uint4 *>(x + i * 16);
        q[1] = *reinterpret_cast<const uint4 *>(x + i * 16 + 8);
        const uint16_t *h = reinterpret_cast<const uint16_t *>(q);
        uint16_t *oh = reinterpret_cast<uint16_t *>(o);
#pragma unroll
        for (int c = 0; c < 16; c++) {
            acc[c] += bf2f(h[c]) * d;
            oh[c] = f2bf(wr[c] * d);
        }
        relu_mask<16>(oh, h);
        acc[16] += d;
        *reinterpret_cast<uint4 *>(dx + i * 16) = o[0];
        *reinterpret_cast<uint4 *>(dx + i * 16 + 8) = o[1];
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int c = 0; c < 17; c++) {
        float v = acc[c];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) red[c][wave] = v;
    }
    __syncthreads();
    if (threadIdx.x < 17)
        part[(size_t)blockIdx.x * 17 + threadIdx.x] =
            (red[threadIdx.x][0] + red[threadIdx.x][1]) + (red[threadIdx.x][2] + red[threadIdx.x][3]);
}

// out[c] = sum over the nrows rows of part[nrows][C] (C <= 128) in row order,
// one workgroup per job.  The sum is one chain of FP32 additions per column
// (its order is part of the result); what it cost was a load latency per
// row, with a launch of one thread per column for each tensor: 593 us per
// bias gradient, 1.44 and 0.61 ms for the head's at 4 x 128^3.  Here the
// workgroup streams the rows through two LDS tiles, the next one's loads in
// flight during the current one's additions, so a row costs an addition, and
// all tensors of a backward pass run side by side in one launch.
constexpr int kSumTile = 8192;   // floats per LDS tile
struct SumRowsJob {
    const float *part;
    float *out;
    int nrows, C;
};
constexpr int kSumRowsJobs = 15;
struct SumRowsArgs {
    SumRowsJob job[kSumRowsJobs];
};
__global__ void __launch_bounds__(256) k_sum_rows(SumRowsArgs a) {
    __shared__ float tile[2][kSumTile];
    const SumRowsJob J = a.job[blockIdx.x];
    const int tid = threadIdx.x, rows = kSumTile / J.C, per = rows * J.C;
    const int64_t total = (int64_t)J.nrows * J.C;
    constexpr int NL = kSumTile / 256;
    float pre[NL];
    auto fetch = [&](int64_t base) {
#pragma unroll
        for (int u = 0; u < NL; u++) {
            const int k = tid + 256 * u;
            pre[u] = k < per && base + k < total ? J.part[base + k] : 0.f;
        }
    };
    float acc = 0.f;
    fetch(0);
    int buf = 0;
    for (int r0 = 0; r0 < J.nrows; r0 += rows, buf ^= 1) {
#pragma unroll
        for (int u = 0; u < NL; u++) tile[buf][tid + 256 * u] = pre[u];
        __syncthreads();   // the other tile's readers were done before the tile before this one was stored
        fetch((int64_t)(r0 + rows) * J.C);
        if (tid < J.C) {
            const float *t = tile[buf] + tid;
            const int n = min(rows, J.nrows - r0);
            int r = 0;
            for (; r + 16 <= n; r += 16) {
                float v[16];
#pragma unroll
                for (int u = 0; u < 16; u++) v[u] = t[(r + u) * J.C];
#pragma unroll
                for (int u = 0; u < 16; u++) acc += v[u];
            }
            for (; r < n; r++) acc += t[r * J.C];
        }
    }
    if (tid < J.C) J.out[tid] = acc;
}

// Partial sums of a [n][C] BF16 tensor (C a power of two, 16..128): partial
// q of nq sums the rows r with (r / L) mod nq = q, L = 256 / C, row class
// r mod L by row class, the classes then in order.  A partial is 32 threads'
// work (a thread takes 8 channels, one 16-byte load, of one row class), a
// workgroup eight partials.
__global__ void __launch_bounds__(256) k_chan_sum_part(const uint16_t *__restrict__ x, int C, int64_t n, int nq,
                                                       float *__restrict__ part) {
    __shared__ float red[256][9];
    const int ng = C >> 3, L = 256 / C;
    const int sub = threadIdx.x >> 5, t32 = threadIdx.x & 31, grp = t32 % ng, r0 = t32 / ng;
    const int q = blockIdx.x * 8 + sub;
    float s[8];
#pragma unroll
    for (int j = 0; j < 8; j++) s[j] = 0.f;
    if (q < nq)
        for (int64_t i = (int64_t)q * L + r0; i < n; i += (int64_t)nq * L) {
            const uint4 w = *reinterpret_cast<const uint4 *>(x + i * C + grp * 8);
            const uint16_t *h = reinterpret_cast<const uint16_t *>(&w);
#pragma unroll
            for (int j = 0; j < 8; j++) s[j] += bf2f(h[j]);
        }
#pragma unroll
    for (int j = 0; j < 8; j++) red[threadIdx.x][j] = s[j];
    __syncthreads();
    for (int k = threadIdx.x; k < 8 * C; k += 256) {
        const int qs = k / C, c = k % C;
        if (blockIdx.x * 8 + qs >= nq) continue;
        float t = 0.f;
        for (int r = 0; r < L; r++) t += red[qs * 32 + r * ng + (c >> 3)][c & 7];
        part[(size_t)(blockIdx.x * 8 + qs) * C + c] = t;
    }
}

// Input features of the network per voxel (8 BF16 channels):
//   0  f / s                       the solve's right-hand side
//   1  phi_s / (s h^2)             the spectral seed (fixed-LOS inverse of f)
//   2  r_s / s                     its residual under the local-LOS operator
//   3  psi / (s h^2)               the fixed-LOS inverse of that residual
//   4-6  rhat - nhat_c             local LOS minus the seed's fixed LOS
//   7  h_ref / |x|                 strength of the first-derivative term
// s = rms(f) of the item (FP64 on the device), h the cell size.
__global__ void k_features(const float *__restrict__ f, const float *__restrict__ phis, const float *__restrict__ rs,
                           const float *__restrict__ psi, const double *__restrict__ ss, FeatArgs a,
                           uint16_t *__restrict__ X) {
    const int nx = 1 << a.lx, ny = 1 << a.ly, nz = 1 << a.lz;
    const int64_t nv = (int64_t)nx * ny * nz;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nv * a.batch;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t item = i / nv;
        const int64_t v = i - item * nv;
        const int x = (int)(v & (nx - 1)), y = (int)((v >> a.lx) & (ny - 1)), z = (int)(v >> (a.lx + a.ly));
        const double s = ss[item] > 0.0 ? ss[item] : 1.0;
        const float inv = (float)(1.0 / s);
        const float px = a.bmin[0] + (x + 0.5f) * a.h[0], py = a.bmin[1] + (y + 0.5f) * a.h[1],
                    pz = a.bmin[2] + (z + 0.5f) * a.h[2];
        const float r = sqrtf(px * px + py * py + pz * pz);
        const float ir = r > 0.f ? 1.f / r : 0.f;
        uint16_t o[8];
        o[0] = f2bf(f[i] * inv);
        o[1] = f2bf(phis[i] * inv * a.ih2);
        o[2] = f2bf(rs[i] * inv);
        o[3] = f2bf(psi[i] * inv * a.ih2);
        o[4] = f2bf(px * ir - a.nc[0]);
        o[5] = f2bf(py * ir - a.nc[1]);
        o[6] = f2bf(pz * ir - a.nc[2]);
        o[7] = f2bf(a.href * ir);
        uint4 q;
        memcpy(&q, o, 16);
        *reinterpret_cast<uint4 *>(X + i * 8) = q;
    }
}

// a += b
__global__ void k_add(float *__restrict__ a, const float *__restrict__ b, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        a[i] += b[i];
}

// target = (phi - phi_s) / (s h^2) and the loss
//   L = (1/N) sum_v sum_a (d(v + e_a) - d(v))^2 / 3,  d = out - target,
// the mean square error of the finite-difference gradient (the displacement
// the seed implies).  dL/dout = -(2 / 3N) lap(d).
__global__ void k_target(const float *__restrict__ phi, const float *__restrict__ phis, const double *__restrict__ ss,
                         float ih2, int64_t nv, int64_t n, float *__restrict__ t) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const double s = ss[i / nv] > 0.0 ? ss[i / nv] : 1.0;
        t[i] = (float)(((double)phi[i] - (double)phis[i]) / s) * ih2;
    }
}
__global__ void __launch_bounds__(256) k_loss(const float *__restrict__ out, const float *__restrict__ t, int lx,
                                              int ly, int lz, int64_t n, float scale, float *__restrict__ dout,
                                              double *__restrict__ part) {
    __shared__ double red[4];
    const int nx = 1 << lx, ny = 1 << ly, nz = 1 << lz;
    const int64_t nv = (int64_t)nx * ny * nz;
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t base = (i / nv) * nv, v = i - base;
        const int x = (int)(v & (nx - 1)), y = (int)((v >> lx) & (ny - 1)), z = (int)(v >> (lx + ly));
        auto d = [&](int xx, int yy, int zz) {
            const int64_t j = base + (((int64_t)(zz & (nz - 1)) * ny + (yy & (ny - 1))) * nx + (xx & (nx - 1)));
            return out[j] - t[j];
        };
        const float d0 = d(x, y, z);
        const float gx = d(x + 1, y, z) - d0, gy = d(x, y + 1, z) - d0, gz = d(x, y, z + 1) - d0;
        acc += (double)gx * gx + (double)gy * gy + (double)gz * gz;
        const float lap = (d(x + 1, y, z) + d(x - 1, y, z) + d(x, y + 1, z) + d(x, y - 1, z) + d(x, y, z + 1) +
                           d(x, y, z - 1)) - 6.f * d0;
        dout[i] = -2.f * scale * lap;
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = ((red[0] + red[1]) + (red[2] + red[3])) * scale;
}

// Adam on the FP32 master copy (bias-corrected step sizes from the host)
__global__ void k_adam(float *__restrict__ w, float *__restrict__ m, float *__restrict__ v,
                       const float *__restrict__ gr, int64_t n, float lr_t, float b1, float b2, float eps,
                       float wd) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float g = gr[i] + wd * w[i];
        const float mi = b1 * m[i] + (1.f - b1) * g;
        const float vi = b2 * v[i] + (1.f - b2) * g * g;
        m[i] = mi;
        v[i] = vi;
        w[i] -= lr_t * mi / (sqrtf(vi) + eps);
    }
}

// the network's output in potential units: out = e s h^2 (add: out += ...)
__global__ void k_apply_seed(const float *__restrict__ e, const double *__restrict__ ss, float h2, int64_t n,
                             int add, float *__restrict__ out) {
    const double s = ss[0] > 0.0 ? ss[0] : 1.0;
    const float k = (float)s * h2;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = add ? out[i] + e[i] * k : e[i] * k;
}

static inline unsigned blocks(int64_t n) {
    int64_t b = (n + 255) / 256;
    return (unsigned)(b > 8192 ? 8192 : (b < 1 ? 1 : b));
}

}  // namespace unet

using namespace unet;

// the layers; and the input gradients that are no layer's shape
#define LAYER_CASES(X)         \
    X(8, 0, 16, false)         \
    X(16, 0, 16, false)        \
    X(16, 0, 32, false)        \
    X(32, 0, 32, false)        \
    X(32, 0, 64, false)        \
    X(64, 0, 64, false)        \
    X(64, 0, 128, false)       \
    X(128, 0, 128, false)      \
    X(64, 128, 64, true)       \
    X(32, 64, 32, true)        \
    X(16, 32, 16, true)
#define CONV_CASES(X)          \
    LAYER_CASES(X)             \
    X(32, 0, 16, false)        \
    X(64, 0, 32, false)        \
    X(128, 0, 64, false)       \
    X(64, 0, 192, false)       \
    X(32, 0, 96, false)        \
    X(16, 0, 48, false)

hipError_t launch_unet_conv(const ConvArgs &a, int c1, int c2, int co, bool relu, bool up2, int batch,
                            hipStream_t s) {
    const int nx = 1 << a.lx, ny = 1 << a.ly, nz = 1 << a.lz;
    // k_conv addresses its inputs with 32-bit element offsets
    const int cmax = c1 > c2 ? c1 : c2;
    if ((int64_t)batch * nx * ny * nz * cmax >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
#define LAUNCH(C1_, C2_, CO_, UP_)                                                                        \
    if (c1 == C1_ && c2 == C2_ && co == CO_ && up2 == UP_) {                                              \
        using T = ConvTile<C1_ + C2_, CO_>;                                                               \
        if (a.mask && !T::maskable(relu)) return hipErrorInvalidValue;                                    \
        const dim3 grid((unsigned)((nx + 15) / 16), (unsigned)((ny + T::MB - 1) / T::MB),                 \
                        (unsigned)((nz + T::ZW - 1) / T::ZW * batch * T::NSPLIT));                        \
        if (relu)                                                                                         \
            hipLaunchKernelGGL((k_conv<C1_, C2_, CO_, true, UP_>), grid, dim3(256), 0, s, a);             \
        else                                                                                              \
            hipLaunchKernelGGL((k_conv<C1_, C2_, CO_, false, UP_>), grid, dim3(256), 0, s, a);            \
        return hipGetLastError();                                                                         \
    }
    CONV_CASES(LAUNCH)
#undef LAUNCH
    return hipErrorInvalidValue;
}

hipError_t launch_unet_wgrad(const WgradArgs &a, int c1, int c2, int co, bool up2, int nchunks, hipStream_t s) {
    // k_conv_wgrad addresses its inputs with 32-bit element offsets
    const int cmax = std::max(std::max(c1, c2), co);
    if (((int64_t)a.batch * cmax << (a.lx + a.ly + a.lz)) >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
    const int cib = (c1 + c2 + 15) / 16, cob = co / (16 * wgrad_nb(co));
    dim3 grid((unsigned)nchunks, (unsigned)(cib * cob));
#define LAUNCH(C1_, C2_, CO_, UP_)                                                                        \
    if (c1 == C1_ && c2 == C2_ && co == CO_ && up2 == UP_) {                                              \
        hipLaunchKernelGGL((k_conv_wgrad<C1_, C2_, CO_, UP_>), grid, dim3(kWgThreads), 0, s, a);          \
        return hipGetLastError();                                                                         \
    }
    LAYER_CASES(LAUNCH)
#undef LAUNCH
    return hipErrorInvalidValue;
}

hipError_t launch_unet_sum_chunks(const float *part, int nch, int64_t n, float *out, hipStream_t s) {
    hipLaunchKernelGGL(k_sum_chunks, dim3(blocks(n)), dim3(256), 0, s, part, nch, n, out);
    return hipGetLastError();
}
hipError_t launch_unet_pack(const float *w, int cin, int co, int transposed, uint16_t *out, hipStream_t s) {
    const int kin = transposed ? co : cin, nout = transposed ? cin : co;
    const int64_t total = (int64_t)((27 * kin + 31) / 32) * (nout / 16) * 512;
    hipLaunchKernelGGL(k_pack, dim3(blocks(total)), dim3(256), 0, s, w, cin, co, transposed, out);
    return hipGetLastError();
}
// lx .. lz: log2 of the fine grid's sides; lc of the channels
hipError_t launch_unet_pool(const uint16_t *in, uint16_t *out, int lx, int ly, int lz, int lc, int batch,
                            hipStream_t s) {
    const int64_t n = ((int64_t)batch << (lx + ly + lz - 3)) << (lc - 3);
    hipLaunchKernelGGL(k_pool, dim3(blocks(n)), dim3(256), 0, s, in, out, lx, ly, lc, n);
    return hipGetLastError();
}
hipError_t launch_unet_pool_bwd(const uint16_t *dc, const uint16_t *y, uint16_t *df, int lx, int ly, int lz, int lc,
                                int batch, hipStream_t s) {
    const int64_t n = ((int64_t)batch << (lx + ly + lz)) << (lc - 3);
    hipLaunchKernelGGL(k_pool_bwd, dim3(blocks(n)), dim3(256), 0, s, dc, y, df, lx, ly, lc, n);
    return hipGetLastError();
}
hipError_t launch_unet_upsample_bwd(const uint16_t *dup, const uint16_t *y, uint16_t *dcoarse, int lx, int ly, int lz,
                                    int lc, int batch, hipStream_t s) {
    const int64_t n = ((int64_t)batch << (lx + ly + lz - 3)) << (lc - 3);
    hipLaunchKernelGGL(k_upsample_bwd, dim3(blocks(n)), dim3(256), 0, s, dup, y, dcoarse, lx, ly, lc, n);
    return hipGetLastError();
}
hipError_t launch_unet_head(const uint16_t *x, const float *w, const float *b, float *out, int64_t n,
                            hipStream_t s) {
    hipLaunchKernelGGL(k_head, dim3(blocks(n)), dim3(256), 0, s, x, w, b, out, n);
    return hipGetLastError();
}
int unet_head_bwd_blocks(int64_t n) { return (int)blocks(n); }
hipError_t launch_unet_head_bwd(const uint16_t *x, const float *w, const float *dout, uint16_t *dx, float *part,
                                int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_head_bwd, dim3(blocks(n)), dim3(256), 0, s, x, w, dout, dx, part, n);
    return hipGetLastError();
}
hipError_t launch_unet_features(const float *f, const float *phis, const float *rs, const float *psi,
                                const double *ss, const FeatArgs &a, uint16_t *X, hipStream_t s) {
    const int64_t n = ((int64_t)a.batch << (a.lx + a.ly + a.lz));
    hipLaunchKernelGGL(k_features, dim3(blocks(n)), dim3(256), 0, s, f, phis, rs, psi, ss, a, X);
    return hipGetLastError();
}
hipError_t launch_add_grid(float *a, const float *b, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_add, dim3(blocks(n)), dim3(256), 0, s, a, b, n);
    return hipGetLastError();
}
hipError_t launch_unet_target(const float *phi, const float *phis, const double *ss, float ih2, int64_t nv, int64_t n,
                              float *t, hipStream_t s) {
    hipLaunchKernelGGL(k_target, dim3(blocks(n)), dim3(256), 0, s, phi, phis, ss, ih2, nv, n, t);
    return hipGetLastError();
}
int unet_loss_blocks(int64_t n) { return (int)blocks(n); }
hipError_t launch_unet_loss(const float *out, const float *t, int lx, int ly, int lz, int64_t n, float scale,
                            float *dout, double *part, hipStream_t s) {
    hipLaunchKernelGGL(k_loss, dim3(blocks(n)), dim3(256), 0, s, out, t, lx, ly, lz, n, scale, dout, part);
    return hipGetLastError();
}
hipError_t launch_unet_adam(float *w, float *m, float *v, const float *g, int64_t n, float lr_t, float b1, float b2,
                            float eps, float wd, hipStream_t s) {
    hipLaunchKernelGGL(k_adam, dim3(blocks(n)), dim3(256), 0, s, w, m, v, g, n, lr_t, b1, b2, eps, wd);
    return hipGetLastError();
}
hipError_t launch_unet_apply_seed(const float *e, const double *ss, float h2, int64_t n, int add, float *out,
                                  hipStream_t s) {
    hipLaunchKernelGGL(k_apply_seed, dim3(blocks(n)), dim3(256), 0, s, e, ss, h2, n, add, out);
    return hipGetLastError();
}

}  // namespace baorec

// ====================================================================== host

namespace baorec {

namespace {
struct LayerDef {
    int c1, c2, co;
    bool up2, relu;
    int level;        // resolution level of the output (0 = finest)
    int in1, in2;     // input activation index (-1: network input X, -2..-4: pooled P0..P2)
};
// The network: levels 0..3 with 16, 32, 64, 128 channels; two 3^3
// convolutions per level on the way down and on the way up, 2x2x2 average
// pooling between levels, nearest upsampling into the decoder, a 1x1 head.
const LayerDef kLayers[14] = {
    {8, 0, 16, false, true, 0, -1, -1},     // 0  e0a
    {16, 0, 16, false, true, 0, 0, -1},     // 1  e0b  (skip 0)
    {16, 0, 32, false, true, 1, -2, -1},    // 2  e1a  (pooled 1)
    {32, 0, 32, false, true, 1, 2, -1},     // 3  e1b  (skip 1)
    {32, 0, 64, false, true, 2, -3, -1},    // 4  e2a
    {64, 0, 64, false, true, 2, 4, -1},     // 5  e2b  (skip 2)
    {64, 0, 128, false, true, 3, -4, -1},   // 6  e3a
    {128, 0, 128, false, true, 3, 6, -1},   // 7  e3b
    {64, 128, 64, true, true, 2, 5, 7},     // 8  d2a  [skip 2 | up e3b]
    {64, 0, 64, false, true, 2, 8, -1},     // 9  d2b
    {32, 64, 32, true, true, 1, 3, 9},      // 10 d1a  [skip 1 | up d2b]
    {32, 0, 32, false, true, 1, 10, -1},    // 11 d1b
    {16, 32, 16, true, true, 0, 1, 11},     // 12 d0a  [skip 0 | up d1b]
    {16, 0, 16, false, true, 0, 12, -1},    // 13 d0b
};
constexpr int kNL = 14;

template <typename T>
hipError_t dalloc(T **p, size_t count) {
    *p = nullptr;
    if (count == 0) count = 1;
    return hipMalloc(reinterpret_cast<void **>(p), sizeof(T) * count);
}
}  // namespace

#define UCHK(x)                              \
    do {                                     \
        hipError_t e_ = (x);                 \
        if (e_ != hipSuccess) return e_;     \
    } while (0)

struct UNet {
    int64_t woff[kNL], boff[kNL], hw = 0, hb = 0, P = 0;
    float *par = nullptr, *grad = nullptr, *am = nullptr, *av = nullptr;
    uint16_t *wp[kNL] = {}, *wpt[kNL] = {};
    int64_t step = 0;
    float h_train = 0.f;
    // activations and gradients of the last forward/backward shape
    int batch = 0, lx = -1, ly = -1, lz = -1;
    uint16_t *X = nullptr, *A[kNL] = {}, *Pl[3] = {}, *dA[kNL] = {}, *dP[3] = {}, *dup[3] = {};
    float *out = nullptr, *dout = nullptr, *wpart = nullptr, *hpart = nullptr, *cpart = nullptr;
    size_t wpart_n = 0;
    size_t cpart_off[kNL] = {};   // each layer's bias-gradient partials in cpart

    UNet() {
        int64_t o = 0;
        for (int i = 0; i < kNL; i++) {
            woff[i] = o;
            o += 27LL * (kLayers[i].c1 + kLayers[i].c2) * kLayers[i].co;
            boff[i] = o;
            o += kLayers[i].co;
        }
        hw = o;
        o += 16;
        hb = o;
        o += 1;
        P = o;
    }
    void free_acts() {
        (void)hipFree(X);
        X = nullptr;
        for (int i = 0; i < kNL; i++) {
            (void)hipFree(A[i]);
            (void)hipFree(dA[i]);
            A[i] = dA[i] = nullptr;
        }
        for (int i = 0; i < 3; i++) {
            (void)hipFree(Pl[i]);
            (void)hipFree(dP[i]);
            (void)hipFree(dup[i]);
            Pl[i] = dP[i] = dup[i] = nullptr;
        }
        (void)hipFree(out);
        (void)hipFree(dout);
        (void)hipFree(hpart);
        (void)hipFree(cpart);
        out = dout = hpart = cpart = nullptr;
        batch = 0;
        lx = ly = lz = -1;
    }
    ~UNet() {
        free_acts();
        (void)hipFree(par);
        (void)hipFree(grad);
        (void)hipFree(am);
        (void)hipFree(av);
        (void)hipFree(wpart);
        for (int i = 0; i < kNL; i++) {
            (void)hipFree(wp[i]);
            (void)hipFree(wpt[i]);
        }
    }
    int64_t nvox(int level) const { return (int64_t)batch << (lx + ly + lz - 3 * level); }

    hipError_t alloc_params() {
        UCHK(dalloc(&par, P));
        UCHK(dalloc(&grad, P));
        UCHK(dalloc(&am, P));
        UCHK(dalloc(&av, P));
        UCHK(hipMemset(am, 0, sizeof(float) * P));
        UCHK(hipMemset(av, 0, sizeof(float) * P));
        UCHK(hipMemset(grad, 0, sizeof(float) * P));
        for (int i = 0; i < kNL; i++) {
            const int cin = kLayers[i].c1 + kLayers[i].c2, co = kLayers[i].co;
            UCHK(dalloc(&wp[i], (size_t)((27 * cin + 31) / 32) * (co / 16) * 512));
            if (i > 0) UCHK(dalloc(&wpt[i], (size_t)((27 * co + 31) / 32) * (cin / 16) * 512));
        }
        return hipSuccess;
    }
    hipError_t pack(hipStream_t s) {
        for (int i = 0; i < kNL; i++) {
            const int cin = kLayers[i].c1 + kLayers[i].c2, co = kLayers[i].co;
            UCHK(launch_unet_pack(par + woff[i], cin, co, 0, wp[i], s));
            if (i > 0) UCHK(launch_unet_pack(par + woff[i], cin, co, 1, wpt[i], s));
        }
        return hipSuccess;
    }
    hipError_t ensure_acts(int b, int x, int y, int z) {
        if (b == batch && x == lx && y == ly && z == lz) return hipSuccess;
        free_acts();
        batch = b;
        lx = x;
        ly = y;
        lz = z;
        UCHK(dalloc(&X, (size_t)nvox(0) * 8));
        for (int i = 0; i < kNL; i++) {
            UCHK(dalloc(&A[i], (size_t)nvox(kLayers[i].level) * kLayers[i].co));
            UCHK(dalloc(&dA[i], (size_t)nvox(kLayers[i].level) * kLayers[i].co));
        }
        for (int l = 0; l < 3; l++) {
            const int c = 16 << l;
            UCHK(dalloc(&Pl[l], (size_t)nvox(l + 1) * c));
            UCHK(dalloc(&dP[l], (size_t)nvox(l + 1) * c));
            UCHK(dalloc(&dup[l], (size_t)nvox(l) * 2 * c));
        }
        UCHK(dalloc(&out, nvox(0)));
        UCHK(dalloc(&dout, nvox(0)));
        UCHK(dalloc(&hpart, (size_t)unet_head_bwd_blocks(nvox(0)) * 17));
        size_t cp = 0;
        for (int i = 0; i < kNL; i++) {
            cpart_off[i] = cp;
            cp += (size_t)chan_parts(nvox(kLayers[i].level)) * kLayers[i].co;
        }
        UCHK(dalloc(&cpart, cp));
        return hipSuccess;
    }
    const uint16_t *input_of(int idx) const {
        if (idx == -1) return X;
        if (idx <= -2) return Pl[-idx - 2];
        return A[idx];
    }
    int lv(int level, int which) const { return (which == 0 ? lx : which == 1 ? ly : lz) - level; }

    hipError_t forward(hipStream_t s) {
        for (int i = 0; i < kNL; i++) {
            const LayerDef &d = kLayers[i];
            ConvArgs a{};
            a.in1 = input_of(d.in1);
            a.in2 = d.in2 >= 0 ? A[d.in2] : nullptr;
            a.w = wp[i];
            a.bias = par + boff[i];
            a.out = A[i];
            a.csplit = d.co;
            a.lx = lv(d.level, 0);
            a.ly = lv(d.level, 1);
            a.lz = lv(d.level, 2);
            UCHK(launch_unet_conv(a, d.c1, d.c2, d.co, d.relu, d.up2, batch, s));
            if (i == 1 || i == 3 || i == 5) {   // pool the skip tensor of this level
                const int l = d.level, lc = 4 + l;
                UCHK(launch_unet_pool(A[i], Pl[l], lv(l, 0), lv(l, 1), lv(l, 2), lc, batch, s));
            }
        }
        return launch_unet_head(A[kNL - 1], par + hw, par + hb, out, nvox(0), s);
    }

    // partials of the per-channel sums of dA[layer] (its bias gradient)
    static int chan_parts(int64_t n);
    hipError_t chan_sum(int layer, hipStream_t s);

    hipError_t backward(hipStream_t s) {
        const int64_t n0 = nvox(0);
        const int hbk = unet_head_bwd_blocks(n0);
        UCHK(launch_unet_head_bwd(A[kNL - 1], par + hw, dout, dA[kNL - 1], hpart, n0, s));
        for (int i = kNL - 1; i >= 0; i--) {
            const LayerDef &d = kLayers[i];
            const int l = d.level;
            const int x = lv(l, 0), y = lv(l, 1), z = lv(l, 2);
            // weight gradient (dA[i] is complete and masked by its ReLU)
            const int cin = d.c1 + d.c2;
            const int64_t nbricks = (int64_t)(((1 << x) + 15) >> 4) * (((1 << y) + 3) >> 2) * (((1 << z) + 3) >> 2) * batch;
            int nch = (int)(nbricks < 256 ? nbricks : 256);
            const int64_t per = (nbricks + nch - 1) / nch;
            nch = (int)((nbricks + per - 1) / per);
            const size_t need = (size_t)nch * 27 * cin * d.co;
            if (need > wpart_n) {
                (void)hipFree(wpart);
                UCHK(dalloc(&wpart, need));
                wpart_n = need;
            }
            WgradArgs g{};
            g.in1 = input_of(d.in1);
            g.in2 = d.in2 >= 0 ? A[d.in2] : nullptr;
            g.dout = dA[i];
            g.part = wpart;
            g.lx = x;
            g.ly = y;
            g.lz = z;
            g.batch = batch;
            g.per = per;
            UCHK(launch_unet_wgrad(g, d.c1, d.c2, d.co, d.up2, nch, s));
            UCHK(launch_unet_sum_chunks(wpart, nch, 27LL * cin * d.co, grad + woff[i], s));
            UCHK(chan_sum(i, s));
            if (i == 0) break;
            // input gradient: the transposed convolution of dA[i]
            ConvArgs a{};
            a.in1 = dA[i];
            a.in2 = nullptr;
            a.w = wpt[i];
            a.bias = nullptr;
            a.lx = x;
            a.ly = y;
            a.lz = z;
            a.csplit = cin;
            if (d.c2 > 0) {   // decoder: [skip | upsampled coarse]
                a.out = dA[d.in1];   // the pooling's part is added, and the mask applied, further down
                a.out2 = dup[l];
                a.csplit = d.c1;
                UCHK(launch_unet_conv(a, d.co, 0, cin, false, false, batch, s));
                UCHK(launch_unet_upsample_bwd(dup[l], A[d.in2], dA[d.in2], x, y, z, 5 + l, batch, s));
            } else if (d.in1 <= -2) {   // encoder input from pooling
                const int pl = -d.in1 - 2;
                a.out = dP[pl];
                UCHK(launch_unet_conv(a, d.co, 0, cin, false, false, batch, s));
                const int sk = 2 * pl + 1;   // the pooled skip layer
                UCHK(launch_unet_pool_bwd(dP[pl], A[sk], dA[sk], lv(pl, 0), lv(pl, 1), lv(pl, 2), 4 + pl, batch, s));
            } else {
                a.out = dA[d.in1];
                a.mask = A[d.in1];
                UCHK(launch_unet_conv(a, d.co, 0, cin, false, false, batch, s));
            }
        }
        return sum_rows(hbk, s);
    }
    // sums the partials of the head's and every layer's bias gradients
    hipError_t sum_rows(int hbk, hipStream_t s);
};

int UNet::chan_parts(int64_t n) { return (int)(n / 64 < 1 ? 1 : (n / 64 > 4096 ? 4096 : n / 64)); }

hipError_t UNet::chan_sum(int layer, hipStream_t s) {
    const LayerDef &d = kLayers[layer];
    const int nq = chan_parts(nvox(d.level));
    hipLaunchKernelGGL(k_chan_sum_part, dim3((unsigned)((nq + 7) / 8)), dim3(256), 0, s, dA[layer], d.co,
                       nvox(d.level), nq, cpart + cpart_off[layer]);
    return hipGetLastError();
}

hipError_t UNet::sum_rows(int hbk, hipStream_t s) {
    SumRowsArgs a{};
    for (int i = 0; i < kNL; i++)
        a.job[i] = {cpart + cpart_off[i], grad + boff[i], chan_parts(nvox(kLayers[i].level)), kLayers[i].co};
    a.job[kNL] = {hpart, grad + hw, hbk, 17};   // the head's 16 weights, then its bias (hb = hw + 16)
    static_assert(kNL + 1 == kSumRowsJobs, "a job per layer and the head");
    hipLaunchKernelGGL(k_sum_rows, dim3(kSumRowsJobs), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace baorec

// ------------------------------------------------------------ C++ interface

namespace baorec {

UNet *unet_create() { return new (std::nothrow) UNet(); }
int64_t unet_count_params() {
    int64_t o = 0;
    for (int i = 0; i < kNL; i++) o += 27LL * (kLayers[i].c1 + kLayers[i].c2) * kLayers[i].co + kLayers[i].co;
    return o + 17;
}
void unet_destroy(UNet *n) { delete n; }
int64_t unet_nparams(const UNet *n) { return n->P; }
float unet_h_train(const UNet *n) { return n->h_train; }
void unet_set_h_train(UNet *n, float h) { n->h_train = h; }
int64_t unet_step(const UNet *n) { return n->step; }

// He-normal convolution weights (std sqrt(2 / fan_in)), zero biases, and a
// head of std 0.01 so that the first outputs are a small correction.
hipError_t unet_init(UNet *n, uint64_t seed, hipStream_t s) {
    if (!n->par) UCHK(n->alloc_params());
    std::vector<float> h((size_t)n->P, 0.f);
    uint64_t st = seed * 0x9E3779B97F4A7C15ull + 0x2545F4914F6CDD1Dull;
    auto next = [&]() {   // splitmix64
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    };
    auto normal = [&]() {   // Box-Muller
        const double u1 = ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0);
        const double u2 = ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0);
        return sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
    };
    for (int i = 0; i < kNL; i++) {
        const int cin = kLayers[i].c1 + kLayers[i].c2;
        const double sd = sqrt(2.0 / (27.0 * cin));
        for (int64_t k = 0; k < 27LL * cin * kLayers[i].co; k++) h[n->woff[i] + k] = (float)(sd * normal());
    }
    for (int c = 0; c < 16; c++) h[n->hw + c] = (float)(0.01 * normal());
    n->step = 0;
    UCHK(hipMemcpyAsync(n->par, h.data(), sizeof(float) * n->P, hipMemcpyHostToDevice, s));
    UCHK(hipMemsetAsync(n->am, 0, sizeof(float) * n->P, s));
    UCHK(hipMemsetAsync(n->av, 0, sizeof(float) * n->P, s));
    UCHK(n->pack(s));
    return hipStreamSynchronize(s);
}

hipError_t unet_set_params(UNet *n, const float *host, hipStream_t s) {
    if (!n->par) UCHK(n->alloc_params());
    UCHK(hipMemcpyAsync(n->par, host, sizeof(float) * n->P, hipMemcpyHostToDevice, s));
    UCHK(hipMemsetAsync(n->am, 0, sizeof(float) * n->P, s));
    UCHK(hipMemsetAsync(n->av, 0, sizeof(float) * n->P, s));
    n->step = 0;
    UCHK(n->pack(s));
    return hipStreamSynchronize(s);
}
hipError_t unet_get_params(const UNet *n, float *host, int grads, hipStream_t s) {
    UCHK(hipMemcpyAsync(host, grads ? n->grad : n->par, sizeof(float) * n->P, hipMemcpyDeviceToHost, s));
    return hipStreamSynchronize(s);
}
bool unet_ready(const UNet *n) { return n && n->par; }

// The input tensor (8 BF16 channels per voxel) of a batch of grids with
// sides 2^lx x 2^ly x 2^lz; allocates the activations for that shape.
hipError_t unet_input(UNet *n, int batch, int lx, int ly, int lz, uint16_t **X) {
    UCHK(n->ensure_acts(batch, lx, ly, lz));
    *X = n->X;
    return hipSuccess;
}
// Device tensor of the last forward/backward (BF16 bits) and its length:
// kind 0 the output of layer i, 1 its gradient after the ReLU mask (what the
// weight and input gradients of layer i used), 2 pooled tensor i (0..2),
// 3 its gradient, 4 the input features.
hipError_t unet_tensor(const UNet *n, int kind, int i, const uint16_t **ptr, int64_t *count) {
    *ptr = nullptr;
    *count = 0;
    if (!n->X) return hipErrorNotReady;
    if ((kind == 0 || kind == 1) && i >= 0 && i < kNL) {
        *ptr = kind == 0 ? n->A[i] : n->dA[i];
        *count = n->nvox(kLayers[i].level) * kLayers[i].co;
    } else if ((kind == 2 || kind == 3) && i >= 0 && i < 3) {
        *ptr = kind == 2 ? n->Pl[i] : n->dP[i];
        *count = n->nvox(i + 1) * (16 << i);
    } else if (kind == 4) {
        *ptr = n->X;
        *count = n->nvox(0) * 8;
    } else {
        return hipErrorInvalidValue;
    }
    return hipSuccess;
}
float *unet_output(UNet *n) { return n->out; }
float *unet_output_grad(UNet *n) { return n->dout; }
hipError_t unet_forward(UNet *n, hipStream_t s) { return n->forward(s); }
hipError_t unet_backward(UNet *n, hipStream_t s) { return n->backward(s); }

hipError_t unet_adam(UNet *n, float lr, hipStream_t s) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    n->step++;
    const double c1 = 1.0 - pow((double)b1, (double)n->step), c2 = 1.0 - pow((double)b2, (double)n->step);
    const float lr_t = (float)(lr * sqrt(c2) / c1);
    UCHK(launch_unet_adam(n->par, n->am, n->av, n->grad, n->P, lr_t, b1, b2, eps, 0.f, s));
    return n->pack(s);
}

}  // namespace baorec
