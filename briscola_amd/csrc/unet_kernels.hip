// HIP kernels of the learned preconditioner: a 3-D convolutional U-Net in
// BF16 with FP32 accumulation on the gfx950 matrix cores.
//
// Activations are channels-last ("NDHWC" with N = 1): element (m, c) of a
// tensor with row stride ld sits at m*ld + c, m = (z*H + y)*W + x.  A
// channel slice of a wider tensor is addressed by (base + offset, ld), which
// is how the U-Net concatenates skip connections without copies.
//
// Convolutions are implicit GEMMs over M = voxels, N = output channels and
// K = 27*Cin (tap-major: k = t*Cin + c, t = (dz+1)*9 + (dy+1)*3 + (dx+1)),
// zero padding at the domain boundary.  Weights are stored [Cout][Kp] with
// Kp = K rounded up to 32 and zero-filled.  The matrix instruction is
// v_mfma_f32_16x16x32_bf16: per wavefront a 16 x 16 FP32 tile of D += A B,
// A 16 x 32 (lane l: row l%16, k = 8*(l/16)..+7), B 32 x 16 (lane l: column
// l%16, k = 8*(l/16)..+7), D (lane l: column l%16, rows 4*(l/16)..+3).
#include "unet_internal.h"

#include <algorithm>

namespace bmg {
namespace unet {

namespace {

typedef __attribute__((__vector_size__(8*sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4*sizeof(float)))) float floatx4;

__device__ __forceinline__ bf16x8 zero8()
{
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = __bf16(0.0f);
    return v;
}

__device__ __forceinline__ float bf2f(bf16 v) { return float(v); }

// Voxel m of a D x H x W grid shifted by tap t; -1 outside the grid.
__device__ __forceinline__ int tap_voxel(const Grid3& g, int z, int y, int x,
                                         int t)
{
    const int dz = t/9 - 1, dy = (t/3) % 3 - 1, dx = t % 3 - 1;
    const int zz = z + dz, yy = y + dy, xx = x + dx;
    if (zz < 0 || zz >= g.D || yy < 0 || yy >= g.H || xx < 0 || xx >= g.W)
        return -1;
    return (zz*g.H + yy)*g.W + xx;
}

// ---------------------------------------------------------------------------
// Forward convolution, 3x3x3 (or 1x1x1 when taps == 1), optional bias and
// ReLU.  A workgroup of 4 wavefronts computes 64 voxels x all output
// channels (NT = Cout/16 tiles per wavefront, Cout <= 192); each wavefront
// owns 16 voxels.  The A fragment (8 consecutive k of one voxel, i.e. 8
// channels of one tap, Cin % 8 == 0) is loaded once per K step and reused
// for every output tile.
template <int NT>
__global__ __launch_bounds__(256) void k_conv_fwd(ConvArgs a)
{
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int M = a.g.D*a.g.H*a.g.W;
    const int m0 = (blockIdx.x*4 + wave)*16;
    if (m0 >= M) return;
    const int row = lane & 15;
    const int kq = (lane >> 4)*8;
    const int m = m0 + row;
    const bool mok = m < M;
    const int x = mok ? m % a.g.W : 0;
    const int y = mok ? (m/a.g.W) % a.g.H : 0;
    const int z = mok ? m/(a.g.W*a.g.H) : 0;
    const int K = a.taps*a.cin;
    floatx4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < a.kp; k0 += 32)
    {
        const int k = k0 + kq;
        bf16x8 av = zero8();
        if (mok && k < K)
        {
            const int t = k/a.cin, c = k - t*a.cin;
            const int v = a.taps == 1 ? m : tap_voxel(a.g, z, y, x, t);
            if (v >= 0)
                av = *reinterpret_cast<const bf16x8*>(a.x + size_t(v)*a.ldx + c);
        }
#pragma unroll
        for (int j = 0; j < NT; j++)
        {
            const int n = j*16 + row;
            const bf16x8 bv = *reinterpret_cast<const bf16x8*>(
                a.w + size_t(n)*a.kp + k);
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc[j], 0,
                                                            0, 0);
        }
    }
    // D: lane holds column n = j*16 + row, voxels m0 + 4*(lane/16) + r
#pragma unroll
    for (int j = 0; j < NT; j++)
    {
        const int n = j*16 + row;
        if (n >= a.cout) continue;
        const float bias = a.bias ? a.bias[n] : 0.0f;
#pragma unroll
        for (int r = 0; r < 4; r++)
        {
            const int mm = m0 + 4*(lane >> 4) + r;
            if (mm >= M) continue;
            float v = acc[j][r] + bias;
            if (a.relu && v < 0.0f) v = 0.0f;
            a.y[size_t(mm)*a.ldy + n] = bf16(v);
        }
    }
}

// LDS-staged forward convolution, 3x3x3.  A workgroup of 4 wavefronts
// computes an output tile of 16 x TY x TZ voxels (x fastest): tile row
// r = 0 .. 4*MT-1 is (y, z) = (r % TY, r / TY) with 16 consecutive x, and
// wavefront w owns rows w*MT .. w*MT+MT-1, one 16-voxel M tile each, times
// all NT output-channel tiles.  The input tile with its one-voxel halo,
// 18 x (TY+2) x (TZ+2) voxels of CH channels, is staged in LDS once per
// channel chunk (CH = Cin when Cin <= 48, else 32-channel chunks, Cin % 32
// == 0), zero outside the domain; every tap's A fragment is then a 16-byte
// LDS read, shared by the NT MFMAs of the M tile, and each B fragment (the
// weights of one k step) is read once per wavefront and shared by its MT
// tiles.  K order within a chunk of all channels: k = t*Cin + c as the
// weights are stored; with chunks, tap-major within the chunk (k = t*Cin +
// chunk*32 + 0..31), the same products summed in another order.
template <int MT>
struct ConvTile {
    static constexpr int TY = MT == 4 ? 8 : (MT == 2 ? 4 : 2);
    static constexpr int TZ = 4*MT/TY;
    static constexpr int HX = 18, HY = TY + 2, HZ = TZ + 2;
    static constexpr int HV = HX*HY*HZ;
};

// CIN > 0: all CIN channels staged at once, the k loop unrolled with each
// step's tap and channel known at compile time per lane group; CIN = 0:
// 32-channel chunks of a runtime channel count (a multiple of 32), the 27
// taps unrolled.  Consecutive k steps alternate between AS accumulator
// sets (2 when the tiles leave registers for it) so that dependent MFMAs do
// not follow each other.
template <int NT, int MT, int CIN, int AS>
__global__ __launch_bounds__(256) void k_conv_fwd_lds(ConvArgs a)
{
    using Tl = ConvTile<MT>;
    constexpr int CH = CIN > 0 ? CIN : 32;
    // LDS voxel stride in elements (padded by 8: 16-byte reads of 16
    // consecutive voxels spread over the banks), known at compile time so
    // that every tap offset is a constant
    constexpr int vs = CH + 8;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    bf16* lds = reinterpret_cast<bf16*>(lds_raw);
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int row = lane & 15;
    const int g = lane >> 4;
    const int kq = g*8;
    const int W = a.g.W, H = a.g.H, D = a.g.D;
    const int ntx = (W + 15)/16, nty = (H + Tl::TY - 1)/Tl::TY;
    const int b = blockIdx.x;
    const int x0 = (b % ntx)*16;
    const int y0 = ((b/ntx) % nty)*Tl::TY;
    const int z0 = (b/(ntx*nty))*Tl::TZ;
    const int nchunk = a.cin/CH;
    const int nb0 = blockIdx.y*NT*16;   // first output channel
    constexpr int parts = CH/8;
    floatx4 acc[AS][MT][NT];
#pragma unroll
    for (int h = 0; h < AS; h++)
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
            acc[h][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    // LDS element offset of this lane's voxel in tile row wave*MT + i (tap
    // offsets 0, the corner of its 3x3x3 stencil in the halo tile)
    int base[MT];
#pragma unroll
    for (int i = 0; i < MT; i++)
    {
        const int r = wave*MT + i;
        base[i] = (((r/Tl::TY)*Tl::HY + r % Tl::TY)*Tl::HX + row)*vs;
    }
    const bf16* wrow[NT];
#pragma unroll
    for (int j = 0; j < NT; j++)
        wrow[j] = a.w + size_t(nb0 + j*16 + row)*a.kp + kq;
    // halo-tile offset of tap t, in voxels
    auto tap_off = [](int t)
    {
        return (t/9)*Tl::HY*Tl::HX + ((t/3) % 3)*Tl::HX + t % 3;
    };
    for (int c0 = 0; c0 < nchunk; c0++)
    {
        if (c0 > 0) __syncthreads();
        for (int u = threadIdx.x; u < Tl::HV*parts; u += 256)
        {
            const int v = u/parts, part = u - v*parts;
            const int hx = v % Tl::HX, hy = (v/Tl::HX) % Tl::HY;
            const int hz = v/(Tl::HX*Tl::HY);
            const int gx = x0 - 1 + hx, gy = y0 - 1 + hy, gz = z0 - 1 + hz;
            bf16x8 val = zero8();
            if (gx >= 0 && gx < W && gy >= 0 && gy < H && gz >= 0 && gz < D)
                val = *reinterpret_cast<const bf16x8*>(
                    a.x + size_t((gz*H + gy)*W + gx)*a.ldx + c0*CH + part*8);
            *reinterpret_cast<bf16x8*>(lds + v*vs + part*8) = val;
        }
        __syncthreads();
        if constexpr (CIN > 0)
        {
            constexpr int K = 27*CIN;
            constexpr int NS = (K + 31)/32;
#pragma unroll
            for (int st = 0; st < NS; st++)
            {
                // this lane group's k = 32 st + 8 g: tap and channel
                int off = -1;
#pragma unroll
                for (int gg = 0; gg < 4; gg++)
                {
                    const int k = st*32 + gg*8;
                    if (k < K && g == gg)
                        off = tap_off(k/CIN)*vs + (k % CIN);
                }
                bf16x8 bv[NT];
#pragma unroll
                for (int j = 0; j < NT; j++)
                    bv[j] = *reinterpret_cast<const bf16x8*>(wrow[j] + st*32);
#pragma unroll
                for (int i = 0; i < MT; i++)
                {
                    bf16x8 av = zero8();
                    if (off >= 0)
                        av = *reinterpret_cast<const bf16x8*>(
                            lds + base[i] + off);
#pragma unroll
                    for (int j = 0; j < NT; j++)
                        acc[st % AS][i][j] =
                            __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                av, bv[j], acc[st % AS][i][j], 0, 0, 0);
                }
            }
        }
        else
        {
#pragma unroll
            for (int t = 0; t < 27; t++)
            {
                const int off = tap_off(t)*vs + kq;
                const int k = t*a.cin + c0*CH;
                bf16x8 bv[NT];
#pragma unroll
                for (int j = 0; j < NT; j++)
                    bv[j] = *reinterpret_cast<const bf16x8*>(wrow[j] + k);
#pragma unroll
                for (int i = 0; i < MT; i++)
                {
                    const bf16x8 av = *reinterpret_cast<const bf16x8*>(
                        lds + base[i] + off);
#pragma unroll
                    for (int j = 0; j < NT; j++)
                        acc[t % AS][i][j] =
                            __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                av, bv[j], acc[t % AS][i][j], 0, 0, 0);
                }
            }
        }
    }
    // D of tile (i, j): lane holds channel n = j*16 + row for the voxels
    // x = x0 + 4*(lane/16) + q, q = 0..3, of tile row wave*MT + i.  Each
    // 16 x 16 tile goes through the wavefront's own 512 bytes of LDS (the
    // input tile is no longer read) so that a lane stores 8 channels of one
    // voxel, 16 bytes; every wavefront passes the same barriers.
    __syncthreads();
    bf16* tb = lds + wave*256;
#pragma unroll
    for (int i = 0; i < MT; i++)
    {
        const int r = wave*MT + i;
        const int yy = y0 + r % Tl::TY, zz = z0 + r/Tl::TY;
#pragma unroll
        for (int j = 0; j < NT; j++)
        {
            const int n = nb0 + j*16 + row;
            const float bias = a.bias ? a.bias[n] : 0.0f;
#pragma unroll
            for (int q = 0; q < 4; q++)
            {
                float v = acc[0][i][j][q] + bias;
                if (AS == 2) v = acc[0][i][j][q] + acc[AS - 1][i][j][q] + bias;
                if (a.relu && v < 0.0f) v = 0.0f;
                tb[(4*g + q)*16 + row] = bf16(v);
            }
            __syncthreads();
            // lanes 0..31: voxel x0 + lane/2, channels nb0 + j*16 + 8*(lane&1)
            if (lane < 32 && yy < H && zz < D)
            {
                const int xx = x0 + (lane >> 1);
                const int n0 = nb0 + j*16 + 8*(lane & 1);
                if (xx < W && n0 < a.cout)
                    *reinterpret_cast<bf16x8*>(
                        a.y + size_t((zz*H + yy)*W + xx)*a.ldy + n0) =
                        *reinterpret_cast<const bf16x8*>(tb + lane*8);
            }
            __syncthreads();
        }
    }
}

// Forward convolution of the inference pass, 3x3x3 with bias and ReLU, input
// channels in chunks of 16: the first c0 of them from a coarse tensor read
// through the nearest-neighbour upsampling, the others from a fine one (the
// skip connection), so neither the upsampled tensor nor the concatenation is
// ever written.  A workgroup of 4 wavefronts owns 16 x TY x TZ voxels and
// 16 NT output channels, a wavefront MT consecutive rows (y) of one plane.
// A chunk's input tile with its halo is staged in LDS as two planes of
// 16-byte units (8 channels of a voxel), so the 16 lanes of a fragment read
// 256 contiguous bytes.  A K step takes 16 channels of two taps with the same
// dy; for a pair of (dz, dx) a wavefront reads the fragments of its MT + 2
// rows once and uses each for the three dy: 10 LDS reads for 24 NT matrix
// instructions (MT = 8), where one read per instruction and output tile had
// the LDS, not the matrix cores, set the time.
// Epilogue through LDS: 16-byte stores; POOL: the 2x2x2 averages of the
// rounded outputs (k_pool8's order) too; HEAD: only the network's 1x1x1
// output projection of them (k_head_fwd's order), cout = 16.
// Summed in another order than the training pass's convolutions (FP32).
// 256^3: 48 -> 16 channels with the upsampling 3.9 ms -> 0.96 ms, 96 -> 32 at
// 128^3 0.94 ms -> 0.57 ms; the whole pass 6.8 -> 2.2 ms.
template <int MT>
struct ConvRows {
    static constexpr int WY = 8/MT;          // wavefronts along y
    static constexpr int TY = 8, TZ = 4/WY;
    static constexpr int HX = 18, HY = TY + 2, HZ = TZ + 2;
    static constexpr int HV = HX*HY*HZ;
    static constexpr int UNITS = 2*HV;
    static constexpr int VOX = 16*TY*TZ;
};

template <int NT, int MT, bool POOL, bool HEAD>
__global__ __launch_bounds__(256) void k_conv_rows(TileConvArgs a)
{
    using Tl = ConvRows<MT>;
    constexpr int OUT = Tl::VOX*NT*2;        // units of the output tile
    // the input tile, and a zero unit for each row of a fragment column
    constexpr int IN = Tl::UNITS + (MT + 1)*Tl::HX + 1;
    constexpr int LDS = IN > OUT ? IN : OUT;
    __shared__ __align__(16) bf16 lds[LDS*8];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = lane & 15, g = lane >> 4;
    const int W = a.g.W, H = a.g.H, D = a.g.D;
    const int ntx = (W + 15)/16, nty = (H + Tl::TY - 1)/Tl::TY;
    const int b = blockIdx.x;
    const int x0 = (b % ntx)*16;
    const int y0 = ((b/ntx) % nty)*Tl::TY;
    const int z0 = (b/(ntx*nty))*Tl::TZ;
    const int nb0 = blockIdx.y*NT*16;
    const int wz = wave/Tl::WY, wy = (wave % Tl::WY)*MT;
    floatx4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    // this lane's half of the channels, and of each tap pair
    const int half = g & 1, second = g >> 1;
    const int base = (half*Tl::HV + (wz*Tl::HY + wy)*Tl::HX + row)*8;
    const bf16* wl = a.w + size_t(nb0 + row)*a.kp + half*8;
    constexpr int PER = (Tl::UNITS + 255)/256;
    bf16x8 pre[PER];
    // unit u of a chunk: voxel u/2 of the halo tile, half u & 1 (16-byte
    // pieces of one voxel in adjacent lanes)
    auto fetch = [&](int ch0)
    {
        const bool coarse = ch0 < a.c0;
#pragma unroll
        for (int k = 0; k < PER; k++)
        {
            const int u = tid + 256*k;
            const int v = u >> 1;
            const int hx = v % Tl::HX, r = v/Tl::HX;
            const int gx = x0 - 1 + hx, gy = y0 - 1 + r % Tl::HY;
            const int gz = z0 - 1 + r/Tl::HY;
            pre[k] = zero8();
            if (u < Tl::UNITS && gx >= 0 && gx < W && gy >= 0 && gy < H &&
                gz >= 0 && gz < D)
            {
                if (coarse)
                    pre[k] = *reinterpret_cast<const bf16x8*>(
                        a.up + size_t(((gz >> 1)*(H >> 1) + (gy >> 1))*
                                      (W >> 1) + (gx >> 1))*a.ldu +
                        ch0 + 8*(u & 1));
                else
                    pre[k] = *reinterpret_cast<const bf16x8*>(
                        a.x + size_t((gz*H + gy)*W + gx)*a.ldx +
                        (ch0 - a.c0) + 8*(u & 1));
            }
        }
    };
    fetch(0);
    if (tid < MT + 2)
        *reinterpret_cast<bf16x8*>(lds + (Tl::UNITS + tid*Tl::HX)*8) = zero8();
    for (int ch0 = 0; ch0 < a.cin; ch0 += 16)
    {
        if (ch0 > 0) __syncthreads();
#pragma unroll
        for (int k = 0; k < PER; k++)
        {
            const int u = tid + 256*k;
            if (u < Tl::UNITS)
                *reinterpret_cast<bf16x8*>(
                    lds + ((u & 1)*Tl::HV + (u >> 1))*8) = pre[k];
        }
        __syncthreads();
        if (ch0 + 16 < a.cin) fetch(ch0 + 16);
#pragma unroll
        for (int q = 0; q < 5; q++)
        {
            // (dz, dx) pairs (0,1), (2,3), (4,5), (6,7), (8,-)
            const int qa = 2*q, qb = q < 4 ? 2*q + 1 : 8;
            const int tq = second ? qb : qa;
            const int dz = tq/3, dx = tq - 3*dz;
            const bool none = q == 4 && second;
            bf16x8 bw[3][NT];
#pragma unroll
            for (int dy = 0; dy < 3; dy++)
#pragma unroll
                for (int j = 0; j < NT; j++)
                {
                    bw[dy][j] = *reinterpret_cast<const bf16x8*>(
                        wl + size_t(j*16)*a.kp + (dz*9 + dy*3 + dx)*a.cin +
                        ch0);
                    if (q == 4 && none) bw[dy][j] = zero8();
                }
            // the missing tap reads zeros: an infinity times a zero weight
            // is a NaN
            const bf16* p = lds + (none ? Tl::UNITS*8
                                        : base + (dz*Tl::HY*Tl::HX + dx)*8);
            bf16x8 av[MT + 2];
#pragma unroll
            for (int r = 0; r < MT + 2; r++)
                av[r] = *reinterpret_cast<const bf16x8*>(p + r*Tl::HX*8);
#pragma unroll
            for (int dy = 0; dy < 3; dy++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            av[i + dy], bw[dy][j], acc[i][j], 0, 0, 0);
        }
    }
    // outputs rounded to BF16 into LDS, [voxel][channel]
    __syncthreads();
    constexpr int NC = 16*NT;
#pragma unroll
    for (int j = 0; j < NT; j++)
    {
        const float bias = a.bias[nb0 + j*16 + row];
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int q = 0; q < 4; q++)
            {
                float v = acc[i][j][q] + bias;
                if (v < 0.0f) v = 0.0f;
                const int vox = (wz*Tl::TY + wy + i)*16 + 4*g + q;
                lds[vox*NC + j*16 + row] = bf16(v);
            }
    }
    __syncthreads();
    if constexpr (HEAD)
    {
        float hw[17];
#pragma unroll
        for (int c = 0; c < 17; c++) hw[c] = a.head[c];
        for (int v = tid; v < Tl::VOX; v += 256)
        {
            const int xx = x0 + (v & 15), yy = y0 + (v >> 4) % Tl::TY;
            const int zz = z0 + (v >> 4)/Tl::TY;
            const bf16x8 lo = *reinterpret_cast<const bf16x8*>(lds + v*16);
            const bf16x8 hi = *reinterpret_cast<const bf16x8*>(lds + v*16 + 8);
            float s = hw[16];
#pragma unroll
            for (int c = 0; c < 8; c++) s += hw[c]*float(lo[c]);
#pragma unroll
            for (int c = 0; c < 8; c++) s += hw[8 + c]*float(hi[c]);
            if (xx < W && yy < H && zz < D)
                a.out[size_t((zz*H + yy)*W + xx)] = s;
        }
    }
    else
    {
        for (int u = tid; u < OUT; u += 256)
        {
            const int part = u % (2*NT), v = u/(2*NT);
            const int xx = x0 + (v & 15), yy = y0 + (v >> 4) % Tl::TY;
            const int zz = z0 + (v >> 4)/Tl::TY;
            if (xx < W && yy < H && zz < D)
                *reinterpret_cast<bf16x8*>(
                    a.y + size_t((zz*H + yy)*W + xx)*a.ldy + nb0 + 8*part) =
                    *reinterpret_cast<const bf16x8*>(lds + u*8);
        }
    }
    if constexpr (POOL)
    {
        for (int u = tid; u < OUT/8; u += 256)
        {
            const int part = u % (2*NT), v = u/(2*NT);
            const int cx = v & 7, cy = (v >> 3) % (Tl::TY/2);
            const int cz = (v >> 3)/(Tl::TY/2);
            float s[8];
#pragma unroll
            for (int q = 0; q < 8; q++) s[q] = 0.0f;
#pragma unroll
            for (int d = 0; d < 8; d++)
            {
                const int vox = ((2*cz + (d >> 2))*Tl::TY + 2*cy +
                                 ((d >> 1) & 1))*16 + 2*cx + (d & 1);
                const bf16x8 t = *reinterpret_cast<const bf16x8*>(
                    lds + vox*NC + 8*part);
#pragma unroll
                for (int q = 0; q < 8; q++) s[q] += float(t[q]);
            }
            bf16x8 o;
#pragma unroll
            for (int q = 0; q < 8; q++) o[q] = bf16(0.125f*s[q]);
            const int X = x0/2 + cx, Y = y0/2 + cy, Z = z0/2 + cz;
            if (X < W/2 && Y < H/2 && Z < D/2)
                *reinterpret_cast<bf16x8*>(
                    a.pool + size_t((Z*(H/2) + Y)*(W/2) + X)*a.ldp + nb0 +
                    8*part) = o;
        }
    }
}

// First convolution of the inference pass from the two FP32 inputs (rounded
// to BF16 as k_pack_input does): 2 -> 16 channels with bias and ReLU, its
// output and the 2x2x2 averages.  K = 9 rows (dz, dy) of three taps times 2
// channels, padded to 8: a lane's values are contiguous in LDS, three matrix
// instructions per 16 voxels where the padding to 8 channels took seven.
__global__ __launch_bounds__(256) void k_conv_first(Grid3 gr, const float* f,
                                                    const float* c,
                                                    const bf16* w, int kp,
                                                    const float* bias, bf16* y,
                                                    int ldy, bf16* pool,
                                                    int ldp)
{
    constexpr int TY = 8, TZ = 4, HX = 18, HY = TY + 2, HZ = TZ + 2;
    constexpr int VOX = 16*TY*TZ;
    __shared__ __align__(16) unsigned char raw[VOX*32];
    // the input tile, then zeros for the rows that are none
    constexpr int ZERO = HX*HY*HZ, ZEROS = (TY - 1)*HX + 3;
    static_assert(VOX*32 >= (ZERO + ZEROS)*4, "");
    unsigned* in = reinterpret_cast<unsigned*>(raw);
    bf16* lds = reinterpret_cast<bf16*>(raw);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 15, g = lane >> 4;
    const int W = gr.W, H = gr.H, D = gr.D;
    const int ntx = (W + 15)/16, nty = (H + TY - 1)/TY;
    const int b = blockIdx.x;
    const int x0 = (b % ntx)*16;
    const int y0 = ((b/ntx) % nty)*TY;
    const int z0 = (b/(ntx*nty))*TZ;
    for (int v = tid; v < HX*HY*HZ; v += 256)
    {
        const int hx = v % HX, r = v/HX;
        const int gx = x0 - 1 + hx, gy = y0 - 1 + r % HY, gz = z0 - 1 + r/HY;
        unsigned two = 0;
        if (gx >= 0 && gx < W && gy >= 0 && gy < H && gz >= 0 && gz < D)
        {
            const size_t m = size_t((gz*H + gy)*W + gx);
            const bf16 p[2] = {bf16(f[m]), bf16(c[m])};
            two = __builtin_bit_cast(unsigned short, p[0]) |
                  (unsigned(__builtin_bit_cast(unsigned short, p[1])) << 16);
        }
        in[v] = two;
    }
    if (tid < ZEROS) in[ZERO + tid] = 0;
    // weights of the lane's output channel, row 4s + g of the nine
    bf16x8 bw[3];
    int off[3];
#pragma unroll
    for (int s = 0; s < 3; s++)
    {
        const int q = 4*s + g;
        bw[s] = zero8();
        if (q < 9)
#pragma unroll
            for (int t = 0; t < 3; t++)
            {
                bw[s][2*t] = w[size_t(row)*kp + (3*q + t)*8];
                bw[s][2*t + 1] = w[size_t(row)*kp + (3*q + t)*8 + 1];
            }
        // past the nine, zeros: an infinity times a zero weight is a NaN
        off[s] = q < 9 ? ((wave + q/3)*HY + q % 3)*HX + row : ZERO;
    }
    __syncthreads();
    floatx4 acc[TY];
#pragma unroll
    for (int i = 0; i < TY; i++)
    {
        acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
        const unsigned* p = in + i*HX;
#pragma unroll
        for (int s = 0; s < 3; s++)
        {
            union { unsigned u[4]; bf16x8 v; } av;
#pragma unroll
            for (int k = 0; k < 3; k++)
                av.u[k] = p[off[s] + k];
            av.u[3] = 0;   // not a neighbour: no value of its may enter
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av.v, bw[s],
                                                            acc[i], 0, 0, 0);
        }
    }
    __syncthreads();
    const float bs = bias[row];
#pragma unroll
    for (int i = 0; i < TY; i++)
#pragma unroll
        for (int q = 0; q < 4; q++)
        {
            float v = acc[i][q] + bs;
            if (v < 0.0f) v = 0.0f;
            lds[((wave*TY + i)*16 + 4*g + q)*16 + row] = bf16(v);
        }
    __syncthreads();
    for (int u = tid; u < VOX*2; u += 256)
    {
        const int v = u >> 1;
        const int xx = x0 + (v & 15), yy = y0 + (v >> 4) % TY;
        const int zz = z0 + (v >> 4)/TY;
        if (xx < W && yy < H && zz < D)
            *reinterpret_cast<bf16x8*>(y + size_t((zz*H + yy)*W + xx)*ldy +
                                       8*(u & 1)) =
                *reinterpret_cast<const bf16x8*>(lds + u*8);
    }
    for (int u = tid; u < VOX/4; u += 256)
    {
        const int part = u & 1, v = u >> 1;
        const int cx = v & 7, cy = (v >> 3) % (TY/2), cz = (v >> 3)/(TY/2);
        float s[8];
#pragma unroll
        for (int q = 0; q < 8; q++) s[q] = 0.0f;
#pragma unroll
        for (int d = 0; d < 8; d++)
        {
            const int vox = ((2*cz + (d >> 2))*TY + 2*cy + ((d >> 1) & 1))*16 +
                            2*cx + (d & 1);
            const bf16x8 t = *reinterpret_cast<const bf16x8*>(lds + vox*16 +
                                                              8*part);
#pragma unroll
            for (int q = 0; q < 8; q++) s[q] += float(t[q]);
        }
        bf16x8 o;
#pragma unroll
        for (int q = 0; q < 8; q++) o[q] = bf16(0.125f*s[q]);
        const int X = x0/2 + cx, Y = y0/2 + cy, Z = z0/2 + cz;
        if (X < W/2 && Y < H/2 && Z < D/2)
            *reinterpret_cast<bf16x8*>(
                pool + size_t((Z*(H/2) + Y)*(W/2) + X)*ldp + 8*part) = o;
    }
}

// Weight gradient dW[n][k] += sum over voxels of dZ[m][n] * X[tap(m)][c] for
// one 16 x 16 tile of (n, k) and one chunk of voxels per wavefront; the
// chunk partial sums are added into the FP32 gradient atomically.
// A = dZ^T (16 n x 32 voxels), B = X_col (32 voxels x 16 k).
__global__ __launch_bounds__(64) void k_conv_wgrad(WgradArgs a)
{
    const int lane = threadIdx.x;
    const int row = lane & 15;
    const int kq = (lane >> 4)*8;
    const int n = blockIdx.y*16 + row;        // A row
    const int kcol = blockIdx.x*16 + row;     // B column
    const int M = a.g.D*a.g.H*a.g.W;
    const int K = a.taps*a.cin;
    const int tcol = kcol < K ? kcol/a.cin : 0;
    const int ccol = kcol < K ? kcol - tcol*a.cin : 0;
    const int mlo = blockIdx.z*a.chunk;
    const int mhi = min(M, mlo + a.chunk);
    floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int mb = mlo; mb < mhi; mb += 32)
    {
        bf16x8 av, bv;
#pragma unroll
        for (int i = 0; i < 8; i++)
        {
            const int m = mb + kq + i;
            bf16 dz = bf16(0.0f), xv = bf16(0.0f);
            if (m < mhi)
            {
                if (n < a.cout) dz = a.dz[size_t(m)*a.lddz + n];
                if (kcol < K)
                {
                    int v = m;
                    if (a.taps != 1)
                    {
                        const int x = m % a.g.W, y = (m/a.g.W) % a.g.H;
                        const int z = m/(a.g.W*a.g.H);
                        v = tap_voxel(a.g, z, y, x, tcol);
                    }
                    if (v >= 0) xv = a.x[size_t(v)*a.ldx + ccol];
                }
            }
            av[i] = dz;
            bv[i] = xv;
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc, 0, 0, 0);
    }
    // D[n][k]: lane holds column k = blockIdx.x*16 + row, rows n = 4*(lane/16)+r
#pragma unroll
    for (int r = 0; r < 4; r++)
    {
        const int nn = blockIdx.y*16 + 4*(lane >> 4) + r;
        if (nn < a.cout && kcol < K)
            atomicAdd(a.dw + size_t(nn)*a.kp + kcol, acc[r]);
    }
}

// Weight gradient of a 3x3x3 convolution from LDS (and the bias gradient,
// the column sums of dZ).  The product reduces over voxels, so its fragments
// hold 8 voxels of one channel, while memory holds the channels of a voxel:
// a tile of X (one voxel of halo) and of dZ is transposed 8x8 in registers on
// its way into LDS.  Along x the tile's 8S positions are grouped by residue
// mod S, x = x0 + r + S e, and a unit is the 16 bytes e = 0..7 of one
// (z, y, r, channel): a tap's shift by +-1 in x is then another residue, and
// residues -1 and S are kept too, so that every fragment is one aligned
// 16-byte read.  A K step of the matrix instruction takes 32 voxels: S
// residues of 4/S planes at one y (S = 4, 2, 1 for rows of at least 17, 9
// and 1 voxels, so that short rows do not multiply zeros).
// A workgroup owns 16 input channels (all 8 of the first layer, two taps per
// 16 columns) and 16 NT output channels for all 27 taps, its four wavefronts
// a quarter of the taps each, the accumulators in registers over all tiles
// of its share; shares are summed by k_wgrad_sum in a fixed order.  Units are
// placed at channel ^ (position & 7), without which the transposed stores hit
// one bank.
// 64^3 training step: one 16x16 tile per wavefront, its fragments gathered
// value by value from memory and added atomically, took 1.5 ms in 7 launches;
// 0.15 ms in this form.
template <int S, int NT, int CC>
struct WgradTile {
    static constexpr int ZG = 4/S;
    static constexpr int YT = NT <= 2 ? 8 : 4;
    static constexpr int XU = (ZG + 2)*(YT + 2)*(S + 2);   // positions of X
    static constexpr int ZU = ZG*YT*S;                     // and dZ
    static constexpr int NN = 16*NT;
    static constexpr int LDS = (XU*CC + ZU*NN)*16;
    static constexpr int BLOCKS = CC == 8 ? 14 : 27;       // of 16 columns
    static constexpr int SLOTS = (BLOCKS + 1 + 3)/4;       // with the bias
};

// Transposes 8 voxels x 8 channels into the units of the 8 channels.
__device__ __forceinline__ void store_units(bf16* lds, int unit0, int sw,
                                            const bf16x8 (&v)[8])
{
#pragma unroll
    for (int c = 0; c < 8; c++)
    {
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = v[e][c];
        *reinterpret_cast<bf16x8*>(lds + 8*(unit0 + (c ^ sw))) = o;
    }
}

template <int S, int NT, int CC>
__global__ __launch_bounds__(256) void k_wgrad_lds(WgradArgs a, int nsplit,
                                                   float* partial)
{
    using Tl = WgradTile<S, NT, CC>;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    bf16* lx = reinterpret_cast<bf16*>(lds_raw);
    bf16* lz = lx + 8*Tl::XU*CC;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 15, g = lane >> 4;
    const int gs = g % S, gz = g/S;
    const int c0 = CC == 8 ? 0 : blockIdx.x*16;
    const int n0 = blockIdx.y*Tl::NN;
    const int W = a.g.W, H = a.g.H, D = a.g.D;
    const int ntx = (W + 8*S - 1)/(8*S), nty = (H + Tl::YT - 1)/Tl::YT;
    const int ntz = (D + Tl::ZG - 1)/Tl::ZG;
    floatx4 acc[Tl::SLOTS][NT];
#pragma unroll
    for (int i = 0; i < Tl::SLOTS; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    bf16x8 ones;
#pragma unroll
    for (int i = 0; i < 8; i++) ones[i] = __bf16(1.0f);
    // position offset of this lane's tap in each slot, and its channel
    int off[Tl::SLOTS];
#pragma unroll
    for (int i = 0; i < Tl::SLOTS; i++)
    {
        const int blk = wave + 4*i;
        const int t = min(CC == 8 ? 2*blk + (row >> 3) : blk, 26);
        off[i] = ((t/9)*(Tl::YT + 2) + (t/3) % 3)*(S + 2) + t % 3;
    }
    const int ch = CC == 8 ? row & 7 : row;
    const int ntiles = ntx*nty*ntz;
    for (int tile = blockIdx.z; tile < ntiles; tile += nsplit)
    {
        const int x0 = (tile % ntx)*8*S;
        const int y0 = ((tile/ntx) % nty)*Tl::YT;
        const int z0 = (tile/(ntx*nty))*Tl::ZG;
        if (tile != int(blockIdx.z)) __syncthreads();
        constexpr int CP = CC/8, NP = Tl::NN/8;
        for (int u = tid; u < Tl::XU*CP; u += 256)
        {
            const int part = u % CP, pos = u/CP;
            const int ss = pos % (S + 2), r = pos/(S + 2);
            const int gy = y0 - 1 + r % (Tl::YT + 2);
            const int gz_ = z0 - 1 + r/(Tl::YT + 2);
            const bool in = gy >= 0 && gy < H && gz_ >= 0 && gz_ < D;
            const bf16* src = a.x + size_t((gz_*H + gy)*W)*a.ldx + c0 + 8*part;
            bf16x8 v[8];
#pragma unroll
            for (int e = 0; e < 8; e++)
            {
                const int gx = x0 - 1 + ss + S*e;
                v[e] = in && gx >= 0 && gx < W
                           ? *reinterpret_cast<const bf16x8*>(
                                 src + ptrdiff_t(gx)*a.ldx)
                           : zero8();
            }
            store_units(lx, pos*CC + 8*part, pos & 7, v);
        }
        for (int u = tid; u < Tl::ZU*NP; u += 256)
        {
            const int part = u % NP, pos = u/NP;
            const int ss = pos % S, r = pos/S;
            const int gy = y0 + r % Tl::YT, gz_ = z0 + r/Tl::YT;
            const bool in = gy < H && gz_ < D;
            const bf16* src = a.dz + size_t((gz_*H + gy)*W)*a.lddz + n0 +
                              8*part;
            bf16x8 v[8];
#pragma unroll
            for (int e = 0; e < 8; e++)
            {
                const int gx = x0 + ss + S*e;
                v[e] = in && gx < W ? *reinterpret_cast<const bf16x8*>(
                                          src + ptrdiff_t(gx)*a.lddz)
                                    : zero8();
            }
            store_units(lz, pos*Tl::NN + 8*part, pos & 7, v);
        }
        __syncthreads();
#pragma unroll 1
        for (int y = 0; y < Tl::YT; y++)
        {
            const int pz = (gz*Tl::YT + y)*S + gs;
            bf16x8 av[NT];
#pragma unroll
            for (int j = 0; j < NT; j++)
                av[j] = *reinterpret_cast<const bf16x8*>(
                    lz + 8*(pz*Tl::NN + ((16*j + row) ^ (pz & 7))));
            const int px = (gz*(Tl::YT + 2) + y)*(S + 2) + gs;
#pragma unroll
            for (int i = 0; i < Tl::SLOTS; i++)
            {
                const int blk = wave + 4*i;
                if (blk > Tl::BLOCKS) continue;
                bf16x8 bv = ones;
                if (blk < Tl::BLOCKS)
                {
                    const int p = px + off[i];
                    bv = *reinterpret_cast<const bf16x8*>(
                        lx + 8*(p*CC + (ch ^ (p & 7))));
                }
#pragma unroll
                for (int j = 0; j < NT; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        av[j], bv, acc[i][j], 0, 0, 0);
            }
        }
    }
    // lane: column blk*16 + row, rows n = 4*(lane/16) + r of tile j
    float* out = partial + size_t(blockIdx.z)*a.cout*(a.kp + 1);
#pragma unroll
    for (int i = 0; i < Tl::SLOTS; i++)
    {
        const int blk = wave + 4*i;
        if (blk > Tl::BLOCKS) continue;
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++)
            {
                const int n = n0 + 16*j + 4*g + r;
                if (blk < Tl::BLOCKS)
                {
                    const int k = CC == 8 ? blk*16 + row
                                          : blk*a.cin + c0 + row;
                    if (k < 27*a.cin) out[size_t(n)*a.kp + k] = acc[i][j][r];
                }
                else if (row == 0 && blockIdx.x == 0)
                    out[size_t(a.cout)*a.kp + n] = acc[i][j][r];
            }
    }
}

// dw[i] += sum of the shares' partials (the bias gradients follow the
// weights'; padding columns are left alone).  64 values per workgroup, four
// groups of shares, summed in a fixed order.
__global__ __launch_bounds__(256) void k_wgrad_sum(const float* partial,
                                                   int nsplit, int cout,
                                                   int kp, int used, int n,
                                                   float* dw)
{
    __shared__ float sm[4][64];
    const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
    const int i = blockIdx.x*64 + lane;
    const size_t stride = size_t(cout)*(kp + 1);
    const bool on = i < n && (i >= cout*kp || i % kp < used);
    float s = 0.0f;
    if (on)
    {
#pragma unroll 8
        for (int k = q; k < nsplit; k += 4) s += partial[k*stride + i];
    }
    sm[q][lane] = s;
    __syncthreads();
    if (q == 0 && on)
        dw[i] += (sm[0][lane] + sm[1][lane]) + (sm[2][lane] + sm[3][lane]);
}

// W'[c][t'*Cout + n] = W[n][(26 - t')*Cin + c]: the weights of the data
// gradient, a forward convolution of dZ with flipped taps and swapped
// channels.
__global__ void k_flip_weights(const bf16* w, int cin, int cout, int kp,
                               int taps, bf16* wt, int kpt)
{
    const int i = blockIdx.x*blockDim.x + threadIdx.x;
    const int total = cin*kpt;
    if (i >= total) return;
    const int c = i/kpt, k = i - c*kpt;
    bf16 v = bf16(0.0f);
    if (k < taps*cout)
    {
        const int t = k/cout, n = k - t*cout;
        const int tsrc = taps == 1 ? 0 : 26 - t;
        v = w[size_t(n)*kp + tsrc*cin + c];
    }
    wt[i] = v;
}

// 2x2x2 average pooling of a channel slice (fine grid g) into a coarse one.
__global__ void k_pool(const bf16* x, int ldx, Grid3 g, int C, bf16* y,
                       int ldy)
{
    const int Dc = g.D/2, Hc = g.H/2, Wc = g.W/2;
    const long i = long(blockIdx.x)*blockDim.x + threadIdx.x;
    if (i >= long(Dc)*Hc*Wc*C) return;
    const int c = int(i % C);
    const int mc = int(i/C);
    const int xc = mc % Wc, yc = (mc/Wc) % Hc, zc = mc/(Wc*Hc);
    float s = 0.0f;
    for (int d = 0; d < 8; d++)
    {
        const int zf = 2*zc + (d >> 2), yf = 2*yc + ((d >> 1) & 1),
                  xf = 2*xc + (d & 1);
        s += bf2f(x[size_t((zf*g.H + yf)*g.W + xf)*ldx + c]);
    }
    y[size_t(mc)*ldy + c] = bf16(0.125f*s);
}

// Gradient of the pooling: every fine voxel receives dY/8 of its parent,
// added to dX (which already holds the skip-connection gradient), times the
// ReLU mask of the fine activation y; 8 channels per thread.
__global__ void k_pool_relu_bwd8(const bf16* dy, int lddy, Grid3 g, int C,
                                 const bf16* y, int ldy, bf16* dx, int lddx)
{
    const int C8 = C/8;
    const long i = long(blockIdx.x)*blockDim.x + threadIdx.x;
    if (i >= long(g.D)*g.H*g.W*C8) return;
    const int c = int(i % C8)*8;
    const int m = int(i/C8);
    const int x = m % g.W, yy = (m/g.W) % g.H, z = m/(g.W*g.H);
    const int mc = ((z/2)*(g.H/2) + yy/2)*(g.W/2) + x/2;
    bf16x8* const out = reinterpret_cast<bf16x8*>(dx + size_t(m)*lddx + c);
    const bf16x8 act = *reinterpret_cast<const bf16x8*>(y + size_t(m)*ldy + c);
    const bf16x8 up = *reinterpret_cast<const bf16x8*>(dy + size_t(mc)*lddy + c);
    const bf16x8 old = *out;
    bf16x8 o;
#pragma unroll
    for (int q = 0; q < 8; q++)
    {
        const float v = float(old[q]) + 0.125f*float(up[q]);
        o[q] = float(act[q]) > 0.0f ? bf16(v) : bf16(0.0f);
    }
    *out = o;
}

// Nearest-neighbour upsampling by 2 of a coarse channel slice into a fine
// one (grid g is the fine grid).
__global__ void k_up(const bf16* x, int ldx, Grid3 g, int C, bf16* y, int ldy)
{
    const long i = long(blockIdx.x)*blockDim.x + threadIdx.x;
    if (i >= long(g.D)*g.H*g.W*C) return;
    const int c = int(i % C);
    const int m = int(i/C);
    const int xx = m % g.W, yy = (m/g.W) % g.H, zz = m/(g.W*g.H);
    const int mc = ((zz/2)*(g.H/2) + yy/2)*(g.W/2) + xx/2;
    y[size_t(m)*ldy + c] = x[size_t(mc)*ldx + c];
}

// k_up and k_pool on 8 channels per thread (16-byte loads and stores;
// C, the row strides and the slice bases multiples of 8 channels), with
// the same per-channel arithmetic.
__global__ void k_up8(const bf16* x, int ldx, Grid3 g, int C, bf16* y,
                      int ldy)
{
    const int C8 = C/8;
    const long i = long(blockIdx.x)*blockDim.x + threadIdx.x;
    if (i >= long(g.D)*g.H*g.W*C8) return;
    const int c = int(i % C8)*8;
    const int m = int(i/C8);
    const int xx = m % g.W, yy = (m/g.W) % g.H, zz = m/(g.W*g.H);
    const int mc = ((zz/2)*(g.H/2) + yy/2)*(g.W/2) + xx/2;
    *reinterpret_cast<bf16x8*>(y + size_t(m)*ldy + c) =
        *reinterpret_cast<const bf16x8*>(x + size_t(mc)*ldx + c);
}

__global__ void k_pool8(const bf16* x, int ldx, Grid3 g, int C, bf16* y,
                        int ldy)
{
    const int Dc = g.D/2, Hc = g.H/2, Wc = g.W/2;
    const int C8 = C/8;
    const long i = long(blockIdx.x)*blockDim.x + threadIdx.x;
    if (i >= long(Dc)*Hc*Wc*C8) return;
    const int c = int(i % C8)*8;
    const int mc = int(i/C8);
    const int xc = mc % Wc, yc = (mc/Wc) % Hc, zc = mc/(Wc*Hc);
    float s[8];
#pragma unroll
    for (int q = 0; q < 8; q++) s[q] = 0.0f;
    for (int d = 0; d < 8; d++)
    {
        const int zf = 2*zc + (d >> 2), yf = 2*yc + ((d >> 1) & 1),
                  xf = 2*xc + (d & 1);
        const bf16x8 v = *reinterpret_cast<const bf16x8*>(
            x + size_t((zf*g.H + yf)*g.W + xf)*ldx + c);
#pragma unroll
        for (int q = 0; q < 8; q++) s[q] += float(v[q]);
    }
    bf16x8 o;
#pragma unroll
    for (int q = 0; q < 8; q++) o[q] = bf16(0.125f*s[q]);
    *reinterpret_cast<bf16x8*>(y + size_t(mc)*ldy + c) = o;
}

// Gradient of the upsampling, the coarse voxel summing its 8 children, times
// the ReLU mask of the coarse activation y, on 8 channels per thread (16-byte
// loads and stores).
__global__ void k_up_relu_bwd8(const bf16* dy, int lddy, Grid3 g, int C,
                               const bf16* y, int ldy, bf16* dx, int lddx)
{
    const int Dc = g.D/2, Hc = g.H/2, Wc = g.W/2, C8 = C/8;
    const long i = long(blockIdx.x)*blockDim.x + threadIdx.x;
    if (i >= long(Dc)*Hc*Wc*C8) return;
    const int c = int(i % C8)*8;
    const int mc = int(i/C8);
    const int xc = mc % Wc, yc = (mc/Wc) % Hc, zc = mc/(Wc*Hc);
    const bf16x8 act = *reinterpret_cast<const bf16x8*>(y + size_t(mc)*ldy + c);
    float s[8];
#pragma unroll
    for (int q = 0; q < 8; q++) s[q] = 0.0f;
#pragma unroll
    for (int d = 0; d < 8; d++)
    {
        const int zf = 2*zc + (d >> 2), yf = 2*yc + ((d >> 1) & 1),
                  xf = 2*xc + (d & 1);
        const bf16x8 v = *reinterpret_cast<const bf16x8*>(
            dy + size_t((zf*g.H + yf)*g.W + xf)*lddy + c);
#pragma unroll
        for (int q = 0; q < 8; q++) s[q] += float(v[q]);
    }
    bf16x8 o;
#pragma unroll
    for (int q = 0; q < 8; q++)
        o[q] = float(act[q]) > 0.0f ? bf16(s[q]) : bf16(0.0f);
    *reinterpret_cast<bf16x8*>(dx + size_t(mc)*lddx + c) = o;
}

// Output projection (1x1x1, 16 channels -> 1, FP32; w[16] is the bias)
// and its gradients.
__global__ void k_head_fwd(const bf16* x, int ldx, int M, const float* w,
                           float* out)
{
    const int m = blockIdx.x*blockDim.x + threadIdx.x;
    if (m >= M) return;
    float s = w[16];
#pragma unroll
    for (int c = 0; c < 16; c++) s += w[c]*bf2f(x[size_t(m)*ldx + c]);
    out[m] = s;
}

// dX[m][c] = g[m] * w[c] where X > 0 (X is a ReLU's output); per-block
// partial sums of g[m]*X[m][c] (16 channels) and of g[m] for the weight and
// bias gradients.
__global__ __launch_bounds__(256) void k_head_bwd(const bf16* x, int ldx,
                                                  int M, const float* w,
                                                  const float* gout,
                                                  bf16* dx, int lddx,
                                                  float* partial)
{
    __shared__ float sm[17][4];
    const int m = blockIdx.x*256 + threadIdx.x;
    float gw[17];
#pragma unroll
    for (int c = 0; c < 17; c++) gw[c] = 0.0f;
    if (m < M)
    {
        const float g = gout[m];
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(
                x + size_t(m)*ldx + 8*h);
            bf16x8 o;
#pragma unroll
            for (int c = 0; c < 8; c++)
            {
                const float xv = float(v[c]);
                gw[8*h + c] = g*xv;
                o[c] = xv > 0.0f ? bf16(g*w[8*h + c]) : bf16(0.0f);
            }
            *reinterpret_cast<bf16x8*>(dx + size_t(m)*lddx + 8*h) = o;
        }
        gw[16] = g;
    }
    // within the wavefront, then the four wavefronts in order
#pragma unroll
    for (int c = 0; c < 17; c++)
    {
        for (int o = 32; o > 0; o >>= 1) gw[c] += __shfl_xor(gw[c], o, 64);
        if ((threadIdx.x & 63) == 0) sm[c][threadIdx.x >> 6] = gw[c];
    }
    __syncthreads();
    if (threadIdx.x < 17)
    {
        const float* v = sm[threadIdx.x];
        partial[size_t(blockIdx.x)*17 + threadIdx.x] =
            (v[0] + v[1]) + (v[2] + v[3]);
    }
}

// Mean-removed squared error: loss partials and the output gradient
// g = 2 (p - t - mean(p - t)) / M, with mean(p - t) = shift.
__global__ __launch_bounds__(256) void k_mse(const float* p, const float* t,
                                             int M, const float* shift,
                                             float* g, float* partial)
{
    __shared__ float sm[256];
    const int m = blockIdx.x*256 + threadIdx.x;
    float e = 0.0f;
    if (m < M)
    {
        const float d = p[m] - t[m] - shift[0];
        g[m] = 2.0f*d/float(M);
        e = d*d;
    }
    sm[threadIdx.x] = e;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1)
    {
        if (int(threadIdx.x) < s) sm[threadIdx.x] += sm[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = sm[0];
}

// Per-block partial sums of a - b (FP32), for the mean shift of the loss.
__global__ __launch_bounds__(256) void k_diff_sum(const float* a,
                                                  const float* b, int M,
                                                  float* partial)
{
    __shared__ float sm[256];
    const int m = blockIdx.x*256 + threadIdx.x;
    sm[threadIdx.x] = m < M ? a[m] - b[m] : 0.0f;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1)
    {
        if (int(threadIdx.x) < s) sm[threadIdx.x] += sm[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = sm[0];
}

// out[c] = scale * sum of column c of a rows x cols FP32 array: one
// workgroup per column, fixed order (one thread per column took 41 us for
// 1024 rows, each addition waiting for its load).
__global__ __launch_bounds__(256) void k_col_sum(const float* in, int rows,
                                                 int cols, float scale,
                                                 float* out)
{
    __shared__ float sm[4];
    const int c = blockIdx.x;
    float s = 0.0f;
#pragma unroll 4
    for (int r = threadIdx.x; r < rows; r += 256) s += in[size_t(r)*cols + c];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[c] = scale*((sm[0] + sm[1]) + (sm[2] + sm[3]));
}

// The BF16 copies of parameter i of the network: the weights [n][k] and, for
// the data gradient, the flipped ones wt[c][t'*cout + n] = w[n][(26-t')*cin +
// c]; biases and the head have none.
__device__ __forceinline__ void refresh_weight(const WeightViews& v, int i,
                                               float w)
{
#pragma unroll
    for (int q = 0; q < WeightViews::LAYERS; q++)
    {
        const WeightView& l = v.l[q];
        const int j = i - l.off;
        if (j < 0 || j >= l.cout*l.kp) continue;
        const bf16 b = bf16(w);
        l.w[j] = b;
        const int n = j/l.kp, k = j - n*l.kp;
        if (l.wt && k < 27*l.cin)
        {
            const int t = k/l.cin, c = k - t*l.cin;
            l.wt[size_t(c)*l.kpt + (26 - t)*l.cout + n] = b;
        }
    }
}

__global__ void k_refresh(WeightViews v, const float* w, int n)
{
    const int i = blockIdx.x*blockDim.x + threadIdx.x;
    if (i < n) refresh_weight(v, i, w[i]);
}

// Adam on the FP32 master weights, with their BF16 copies.
__global__ void k_adam(WeightViews views, float* w, float* mo, float* ve,
                       const float* g, int n, float lr, float b1, float b2,
                       float eps, float c1, float c2)
{
    const int i = blockIdx.x*blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float m = b1*mo[i] + (1.0f - b1)*gi;
    const float v = b2*ve[i] + (1.0f - b2)*gi*gi;
    mo[i] = m;
    ve[i] = v;
    const float wi = w[i] - lr*(m/c1)/(sqrtf(v/c2) + eps);
    w[i] = wi;
    refresh_weight(views, i, wi);
}

// Network input from the solver's FP64 colour-split level-0 fields is built
// on the host side of this module (input channels: scaled right-hand side,
// scaled log coefficient, zero padding to 8).
__global__ void k_pack_input(const float* f, const float* lam, int M,
                             bf16* x)
{
    const int m = blockIdx.x*blockDim.x + threadIdx.x;
    if (m >= M) return;
    x[size_t(m)*8 + 0] = bf16(f[m]);
    x[size_t(m)*8 + 1] = bf16(lam[m]);
#pragma unroll
    for (int c = 2; c < 8; c++) x[size_t(m)*8 + c] = bf16(0.0f);
}

inline unsigned nblk(long n, int b) { return unsigned((n + b - 1)/b); }

}  // namespace

namespace {

template <int NT, int MT, int CIN, int AS>
void launch_conv_lds(const ConvArgs& a, hipStream_t s, int groups = 1)
{
    using Tl = ConvTile<MT>;
    const int ch = CIN > 0 ? CIN : 32;
    const int vs = ch + 8;
    const size_t shm = size_t(Tl::HV)*vs*sizeof(bf16);
    const unsigned nb = unsigned((a.g.W + 15)/16)*
                        unsigned((a.g.H + Tl::TY - 1)/Tl::TY)*
                        unsigned((a.g.D + Tl::TZ - 1)/Tl::TZ);
    hipLaunchKernelGGL((k_conv_fwd_lds<NT, MT, CIN, AS>), dim3(nb, groups),
                       dim3(256), shm, s, a);
}

template <int NT, int CIN>
void conv_lds_mt(const ConvArgs& a, hipStream_t s)
{
    constexpr int MT0 = NT <= 4 ? 4 : (NT <= 8 ? 2 : 1);
    constexpr int ch = CIN > 0 ? CIN : 32;
    constexpr bool fit4 = ConvTile<4>::HV*(ch + 8)*2 <= 65536;
    constexpr bool fit2 = ConvTile<2>::HV*(ch + 8)*2 <= 65536;
    constexpr int MT = (MT0 >= 4 && fit4) ? 4 : ((MT0 >= 2 && fit2) ? 2 : 1);
    constexpr int AS = NT*MT <= 8 ? 2 : 1;
    using Tl = ConvTile<MT>;
    const long nb = long((a.g.W + 15)/16)*((a.g.H + Tl::TY - 1)/Tl::TY)*
                    ((a.g.D + Tl::TZ - 1)/Tl::TZ);
    if (nb < 256 && (MT > 1 || NT > 2))
    {
        // a small grid fills too few of the 256 compute units with large
        // tiles: 64 voxels by 16 or 32 channels per workgroup, the k steps
        // summed as the large tile sums them (192 -> 64 channels at 16^3: 16
        // workgroups 106 us, 128 workgroups 35 us)
        if (NT % 2 == 0)
            launch_conv_lds<2, 1, CIN, AS>(a, s, NT/2);
        else
            launch_conv_lds<1, 1, CIN, AS>(a, s, NT);
        return;
    }
    launch_conv_lds<NT, MT, CIN, AS>(a, s);
}

// Output tiles per wavefront: at most 16 accumulator tiles (NT x MT), and
// a staged input tile within 64 KB of LDS (measured: Cin = 48 with four M
// tiles per wavefront in 80 KB was slower than two in 48 KB).
template <int NT>
void conv_lds(const ConvArgs& a, hipStream_t s)
{
    switch (a.cin)
    {
    case 8: conv_lds_mt<NT, 8>(a, s); return;
    case 16: conv_lds_mt<NT, 16>(a, s); return;
    case 32: conv_lds_mt<NT, 32>(a, s); return;
    case 48: conv_lds_mt<NT, 48>(a, s); return;
    default: conv_lds_mt<NT, 0>(a, s); return;
    }
}

}  // namespace

void conv_fwd(const ConvArgs& a, hipStream_t s)
{
    const int M = a.g.D*a.g.H*a.g.W;
    const dim3 g(nblk(M, 64));
    if (a.cout % 16 || a.cin % 8 || a.ldx % 8 || a.kp % 32)
        throw UnetError("convolution shape not supported");
    if (a.taps == 27 && (a.cin == 8 || a.cin == 16 || a.cin == 48 ||
                         a.cin % 32 == 0))
    {
        switch (a.cout/16)
        {
        case 1: conv_lds<1>(a, s); return;
        case 2: conv_lds<2>(a, s); return;
        case 3: conv_lds<3>(a, s); return;
        case 4: conv_lds<4>(a, s); return;
        case 6: conv_lds<6>(a, s); return;
        case 8: conv_lds<8>(a, s); return;
        case 12: conv_lds<12>(a, s); return;
        default: throw UnetError("unsupported output channel count");
        }
    }
    switch (a.cout/16)
    {
    case 1: hipLaunchKernelGGL((k_conv_fwd<1>), g, dim3(256), 0, s, a); break;
    case 2: hipLaunchKernelGGL((k_conv_fwd<2>), g, dim3(256), 0, s, a); break;
    case 3: hipLaunchKernelGGL((k_conv_fwd<3>), g, dim3(256), 0, s, a); break;
    case 4: hipLaunchKernelGGL((k_conv_fwd<4>), g, dim3(256), 0, s, a); break;
    case 6: hipLaunchKernelGGL((k_conv_fwd<6>), g, dim3(256), 0, s, a); break;
    case 8: hipLaunchKernelGGL((k_conv_fwd<8>), g, dim3(256), 0, s, a); break;
    case 12: hipLaunchKernelGGL((k_conv_fwd<12>), g, dim3(256), 0, s, a); break;
    default: throw UnetError("unsupported output channel count");
    }
}

namespace {

template <int NT, int MT>
void launch_rows(const TileConvArgs& a, hipStream_t s)
{
    using Tl = ConvRows<MT>;
    const dim3 g(unsigned((a.g.W + 15)/16)*
                     unsigned((a.g.H + Tl::TY - 1)/Tl::TY)*
                     unsigned((a.g.D + Tl::TZ - 1)/Tl::TZ),
                 unsigned(a.cout/(16*NT)));
    if (a.head)
    {
        if constexpr (NT == 1)
            hipLaunchKernelGGL((k_conv_rows<NT, MT, false, true>), g,
                               dim3(256), 0, s, a);
    }
    else if (a.pool)
        hipLaunchKernelGGL((k_conv_rows<NT, MT, true, false>), g, dim3(256), 0,
                           s, a);
    else
        hipLaunchKernelGGL((k_conv_rows<NT, MT, false, false>), g, dim3(256),
                           0, s, a);
}

}  // namespace

void conv_rows(const TileConvArgs& a, hipStream_t s, int nt, int mt)
{
    if (a.cin % 16 || a.c0 % 16 || a.cout % 16 || a.ldx % 8 || a.ldu % 8 ||
        a.ldy % 8 || a.ldp % 8 || a.kp % 8 || (a.head && a.cout != 16))
        throw UnetError("convolution shape not supported");
    // the largest tile that gives two workgroups per compute unit (512):
    // 512 voxels (mt 8) by 64 channels, 256 by 64, 512 by 32, 512 by 16;
    // below that 256 voxels by 16 channels
    const long big = long((a.g.W + 15)/16)*((a.g.H + 7)/8)*((a.g.D + 3)/4);
    if (nt == 0)
    {
        nt = 1;
        mt = 8;
        if (a.cout % 64 == 0 && big*(a.cout/64) >= 512)
            nt = 4;
        else if (a.cout % 64 == 0 && 2*big*(a.cout/64) >= 512)
            nt = mt = 4;
        else if (a.cout % 32 == 0 && big*(a.cout/32) >= 512)
            nt = 2;
        else if (big*(a.cout/16) < 512)
            mt = 4;
    }
    auto tile = [&](int n, int m)
    {
        return nt == n && mt == m && a.cout % (16*n) == 0;
    };
    if (tile(4, 8))
        launch_rows<4, 8>(a, s);
    else if (tile(4, 4))
        launch_rows<4, 4>(a, s);
    else if (tile(2, 8))
        launch_rows<2, 8>(a, s);
    else if (tile(1, 8))
        launch_rows<1, 8>(a, s);
    else if (tile(1, 4))
        launch_rows<1, 4>(a, s);
    else
        throw UnetError("convolution tile not supported");
}

void conv_first(const Grid3& g, const float* f, const float* c, const bf16* w,
                int kp, const float* bias, bf16* y, int ldy, bf16* pool,
                int ldp, hipStream_t s)
{
    const unsigned n = unsigned((g.W + 15)/16)*unsigned((g.H + 7)/8)*
                       unsigned((g.D + 3)/4);
    hipLaunchKernelGGL(k_conv_first, dim3(n), dim3(256), 0, s, g, f, c, w, kp,
                       bias, y, ldy, pool, ldp);
}

namespace {

template <int S, int NT, int CC>
int wgrad_lds(const WgradArgs& a, int nsplit, float* partial, hipStream_t s)
{
    using Tl = WgradTile<S, NT, CC>;
    static_assert(Tl::LDS <= 65536, "tile exceeds 64 KB of LDS");
    const int ntiles = ((a.g.W + 8*S - 1)/(8*S))*
                       ((a.g.H + Tl::YT - 1)/Tl::YT)*
                       ((a.g.D + Tl::ZG - 1)/Tl::ZG);
    const int gx = CC == 8 ? 1 : a.cin/16, gy = a.cout/Tl::NN;
    // about two workgroups per compute unit
    const int n = std::max(1, std::min({ntiles, nsplit, 512/(gx*gy)}));
    hipLaunchKernelGGL((k_wgrad_lds<S, NT, CC>), dim3(gx, gy, n), dim3(256),
                       Tl::LDS, s, a, n, partial);
    return n;
}

template <int S, int NT>
int wgrad_cc(const WgradArgs& a, int nsplit, float* partial, hipStream_t s)
{
    return a.cin == 8 ? wgrad_lds<S, NT, 8>(a, nsplit, partial, s)
                      : wgrad_lds<S, NT, 16>(a, nsplit, partial, s);
}

template <int S>
int wgrad_nt(const WgradArgs& a, int nsplit, float* partial, hipStream_t s)
{
    if (a.cout % 64 == 0) return wgrad_cc<S, 4>(a, nsplit, partial, s);
    if (a.cout % 32 == 0) return wgrad_cc<S, 2>(a, nsplit, partial, s);
    return wgrad_cc<S, 1>(a, nsplit, partial, s);
}

}  // namespace

size_t wgrad_workspace(const WgradArgs& a)
{
    const bool tiled = a.taps == 27 && (a.cin == 8 || a.cin % 16 == 0) &&
                       a.cout % 16 == 0 && a.ldx % 8 == 0 &&
                       a.lddz % 8 == 0 &&
                       reinterpret_cast<uintptr_t>(a.x) % 16 == 0 &&
                       reinterpret_cast<uintptr_t>(a.dz) % 16 == 0;
    if (!tiled) return 0;
    // at most 512 workgroups, one share each, and no more shares than tiles
    const int S = a.g.W > 16 ? 4 : (a.g.W > 8 ? 2 : 1);
    const int nt = a.cout % 64 == 0 ? 4 : (a.cout % 32 == 0 ? 2 : 1);
    const int yt = nt <= 2 ? 8 : 4, zg = 4/S;
    const long tiles = long((a.g.W + 8*S - 1)/(8*S))*((a.g.H + yt - 1)/yt)*
                       ((a.g.D + zg - 1)/zg);
    const int groups = (a.cin == 8 ? 1 : a.cin/16)*(a.cout/(16*nt));
    const long n = std::max(1L, std::min(tiles, long(512/groups)));
    return size_t(n)*a.cout*(a.kp + 1);
}

// Shapes and alignments the tiled kernel takes (wgrad_workspace > 0) go to
// it; any other goes to the general one (its bias gradient is then the
// caller's).
void conv_wgrad(const WgradArgs& a, float* workspace, float* dbias,
                hipStream_t s)
{
    const size_t need = wgrad_workspace(a);
    if (need && workspace)
    {
        const int S = a.g.W > 16 ? 4 : (a.g.W > 8 ? 2 : 1);
        const int nsplit = int(need/(size_t(a.cout)*(a.kp + 1)));
        const int n = S == 4 ? wgrad_nt<4>(a, nsplit, workspace, s)
                    : (S == 2 ? wgrad_nt<2>(a, nsplit, workspace, s)
                              : wgrad_nt<1>(a, nsplit, workspace, s));
        // dbias, when asked for, follows the weights
        const int total = a.cout*a.kp + (dbias ? a.cout : 0);
        if (dbias && dbias != a.dw + size_t(a.cout)*a.kp)
            throw UnetError("bias gradient must follow the weights'");
        hipLaunchKernelGGL(k_wgrad_sum, dim3(nblk(total, 64)), dim3(256), 0, s,
                           workspace, n, a.cout, a.kp, 27*a.cin, total, a.dw);
        return;
    }
    if (dbias || a.chunk < 1)
        throw UnetError("weight gradient shape not supported");
    const int M = a.g.D*a.g.H*a.g.W;
    const int K = a.taps*a.cin;
    const dim3 g(nblk(K, 16), nblk(a.cout, 16), nblk(M, a.chunk));
    hipLaunchKernelGGL(k_conv_wgrad, g, dim3(64), 0, s, a);
}

void flip_weights(const bf16* w, int cin, int cout, int kp, int taps, bf16* wt,
                  int kpt, hipStream_t s)
{
    hipLaunchKernelGGL(k_flip_weights, dim3(nblk(long(cin)*kpt, 256)),
                       dim3(256), 0, s, w, cin, cout, kp, taps, wt, kpt);
}

void pool(const bf16* x, int ldx, Grid3 g, int C, bf16* y, int ldy,
          hipStream_t s)
{
    const long n = long(g.D/2)*(g.H/2)*(g.W/2)*C;
    if (C % 8 == 0 && ldx % 8 == 0 && ldy % 8 == 0 &&
        reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
        reinterpret_cast<uintptr_t>(y) % 16 == 0)
        hipLaunchKernelGGL(k_pool8, dim3(nblk(n/8, 256)), dim3(256), 0, s, x,
                           ldx, g, C, y, ldy);
    else
        hipLaunchKernelGGL(k_pool, dim3(nblk(n, 256)), dim3(256), 0, s, x,
                           ldx, g, C, y, ldy);
}

void pool_relu_bwd(const bf16* dy, int lddy, Grid3 g, int C, const bf16* y,
                   int ldy, bf16* dx, int lddx, hipStream_t s)
{
    const long n = long(g.D)*g.H*g.W*C/8;
    hipLaunchKernelGGL(k_pool_relu_bwd8, dim3(nblk(n, 256)), dim3(256), 0, s,
                       dy, lddy, g, C, y, ldy, dx, lddx);
}

void up(const bf16* x, int ldx, Grid3 g, int C, bf16* y, int ldy,
        hipStream_t s)
{
    const long n = long(g.D)*g.H*g.W*C;
    if (C % 8 == 0 && ldx % 8 == 0 && ldy % 8 == 0 &&
        reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
        reinterpret_cast<uintptr_t>(y) % 16 == 0)
        hipLaunchKernelGGL(k_up8, dim3(nblk(n/8, 256)), dim3(256), 0, s, x, ldx,
                           g, C, y, ldy);
    else
        hipLaunchKernelGGL(k_up, dim3(nblk(n, 256)), dim3(256), 0, s, x, ldx, g,
                           C, y, ldy);
}

void up_relu_bwd(const bf16* dy, int lddy, Grid3 g, int C, const bf16* y,
                 int ldy, bf16* dx, int lddx, hipStream_t s)
{
    const long n = long(g.D/2)*(g.H/2)*(g.W/2)*C/8;
    hipLaunchKernelGGL(k_up_relu_bwd8, dim3(nblk(n, 256)), dim3(256), 0, s, dy,
                       lddy, g, C, y, ldy, dx, lddx);
}

void head_fwd(const bf16* x, int ldx, int M, const float* w, float* out,
              hipStream_t s)
{
    hipLaunchKernelGGL(k_head_fwd, dim3(nblk(M, 256)), dim3(256), 0, s, x, ldx,
                       M, w, out);
}

int head_bwd(const bf16* x, int ldx, int M, const float* w, const float* gout,
             bf16* dx, int lddx, float* partial, hipStream_t s)
{
    const unsigned nb = nblk(M, 256);
    hipLaunchKernelGGL(k_head_bwd, dim3(nb), dim3(256), 0, s, x, ldx, M, w,
                       gout, dx, lddx, partial);
    return int(nb);
}

int mse(const float* p, const float* t, int M, const float* shift, float* g,
        float* partial, hipStream_t s)
{
    const unsigned nb = nblk(M, 256);
    hipLaunchKernelGGL(k_mse, dim3(nb), dim3(256), 0, s, p, t, M, shift, g,
                       partial);
    return int(nb);
}

int diff_sum(const float* a, const float* b, int M, float* partial,
             hipStream_t s)
{
    const unsigned nb = nblk(M, 256);
    hipLaunchKernelGGL(k_diff_sum, dim3(nb), dim3(256), 0, s, a, b, M, partial);
    return int(nb);
}

void col_sum(const float* in, int rows, int cols, float scale, float* out,
             hipStream_t s)
{
    hipLaunchKernelGGL(k_col_sum, dim3(cols), dim3(256), 0, s, in, rows, cols,
                       scale, out);
}

void adam(const WeightViews& views, float* w, float* m, float* v,
          const float* g, int n, float lr, float b1, float b2, float eps,
          int step, hipStream_t s)
{
    const float c1 = 1.0f - powf(b1, float(step));
    const float c2 = 1.0f - powf(b2, float(step));
    hipLaunchKernelGGL(k_adam, dim3(nblk(n, 256)), dim3(256), 0, s, views, w,
                       m, v, g, n, lr, b1, b2, eps, c1, c2);
}

void refresh_weights(const WeightViews& views, const float* w, int n,
                     hipStream_t s)
{
    hipLaunchKernelGGL(k_refresh, dim3(nblk(n, 256)), dim3(256), 0, s, views,
                       w, n);
}

void pack_input(const float* f, const float* lam, int M, bf16* x,
                hipStream_t s)
{
    hipLaunchKernelGGL(k_pack_input, dim3(nblk(M, 256)), dim3(256), 0, s, f,
                       lam, M, x);
}

}  // namespace unet
}  // namespace bmg
