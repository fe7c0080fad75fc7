// Learned closure: a three-layer 3x3x3 convolutional network (5 -> 32 -> 32
// -> 5 channels, ReLU between layers) that maps the coarse state after a
// time step to a correction of it, trained against box-filtered fine-grid
// runs.  It has no counterpart in the reference; the compact filter stays in
// every step, so a context without a network is the plain scheme.
//
// Every convolution is an implicit GEMM on the gfx950 BF16 matrix cores
// (v_mfma_f32_32x32x16_bf16, FP32 accumulate), its input halo staged in LDS
// and its weights held in registers; activations are BF16 channel-last
// [voxel][channel].
//   forward        out[v][o]  = sum_{t,c} a[nb(v,t)][c] W[o][t][c] (+ b[o])
//   data gradient  g[v][c]    = sum_{t,o} go[nb(v,t)][o] W[o][26-t][c]
//   weight grad.   gW[o][t][c] = sum_v go[v][o] a[nb(v,t)][c]   (partial sums
//                  per workgroup of voxel tiles, then summed in a fixed order)
// Parameters are FP32 (Adam); the update writes their BF16 copies in the
// order in which the kernels' lanes hold them.  The grid is periodic, n^3
// voxels (the context's stored duplicate planes are filled from their
// originals).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <random>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/cnd.h"
#include "cnd_internal.hpp"

using namespace cnd;

namespace {

using bf16 = unsigned short;   // bfloat16 bit pattern
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int kC0 = 5, kC0P = 8, kC1 = 32, kC2 = 32, kC3 = 5, kCP = 32, kTaps = 27;
// flat FP32 parameters: W1 [32][27][5], b1 [32], W2 [32][27][32], b2 [32],
// W3 [5][27][32], b3 [5]
constexpr int kOW1 = 0, kOB1 = kOW1 + kC1 * kTaps * kC0, kOW2 = kOB1 + kC1, kOB2 = kOW2 + kC2 * kTaps * kC1,
              kOW3 = kOB2 + kC2, kOB3 = kOW3 + kC3 * kTaps * kC2, kNParam = kOB3 + kC3;
// one workgroup's weight gradients: layer 2 [tap][4][64 lanes][4], layer 3
// [tap][64][4] (8 output channels), layer 1 [column tile][4][64][4]
constexpr int kP2 = kTaps * 1024, kP3 = kTaps * 256, kP1 = 7 * 1024;
// a slice of the summed gradients: layers 2, 1, 3, then their biases
constexpr int kS2 = 0, kS1 = kP2, kS3 = kS1 + kP1, kSB1 = kS3 + kP3, kSB2 = kSB1 + kCP, kSB3 = kSB2 + kCP,
              kSlice = kSB3 + kCP;
constexpr int kWgSlices = 8;            // slices of the first reduction level

__host__ __device__ inline uint32_t f2u(float f)
{
    union { float f; uint32_t u; } x;
    x.f = f;
    return x.u;
}
__host__ __device__ inline float u2f(uint32_t u)
{
    union { float f; uint32_t u; } x;
    x.u = u;
    return x.f;
}
// round to nearest even
__host__ __device__ inline bf16 to_bf16(float f)
{
    uint32_t u = f2u(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return bf16((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);
    return bf16(u >> 16);
}
__host__ __device__ inline float from_bf16(bf16 h) { return u2f(uint32_t(h) << 16); }

// a modulo n for -n <= a < 2 n: of a, a + n and a - n the one in range is the
// smallest as an unsigned number
__device__ __forceinline__ int wrap(int a, int n)
{
    const unsigned b = min(unsigned(a), unsigned(a + n));
    return int(min(b, b - unsigned(n)));
}
typedef short s8v __attribute__((ext_vector_type(8)));
typedef short s4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4v *lds_s4;

__device__ __forceinline__ f16v mfma16(const s8v &a, const s8v &b, const f16v &c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8v, a), __builtin_bit_cast(bf8v, b), c, 0, 0,
                                                  0);
}

// four values rounded to BF16 (nearest even, as to_bf16; v_cvt_pk_bf16_f32)
__device__ __forceinline__ s4v pack4(const float (&x)[4])
{
    typedef __bf16 b4v __attribute__((ext_vector_type(4)));
    b4v b;
#pragma unroll
    for (int k = 0; k < 4; ++k) b[k] = __bf16(x[k]);
    return __builtin_bit_cast(s4v, b);
}

// x extent of a wave's 32 voxels for an n^3 grid (n a multiple of 8)
__host__ inline int conv_x(int n) { return n % 32 == 0 ? 32 : (n % 16 == 0 ? 16 : 8); }

// Tiles of a workgroup: each XCD (blockIdx.x % 8) takes a contiguous eighth of
// the tiles, a slab of the grid whose halos its L2 then holds (64^3, 32
// channels: 2 MB of 4), and its workgroups, `rank` of `ranks`, walk it together.
struct Walk {
    int first, end, step;
    __device__ Walk(int ntiles, int rank, int ranks)
    {
        const int per = (ntiles + 7) / 8, a = int(blockIdx.x % 8) * per;
        first = a + rank;
        end = min(a + per, ntiles);
        step = ranks;
    }
};

// What a convolution reads and writes besides its input: FWD, BF16 [V][32]
// out = ReLU(acc + bias); OUT, FP32 [V][5] out = acc (+ bias); MASK, BF16
// [V][32] out = acc where mask > 0, else 0; LOSS, the mean-square loss of
// y = acc + bias against the FP32 [V][5] target tg: each workgroup's sum of
// (y - tg)^2 to lpart and, with out, its gradient 2 (y - tg) / (5 V) as BF16
// [V][8] (channels 5.. zero).
enum Epi { FWD, OUT, MASK, LOSS };
// How K = 16 of an instruction is filled: C32, half the 32 channels of one
// tap; PAIR, the 8 channels of two taps (lanes kh = 0 and 1; the 28th tap is
// zero); SINGLE, the 8 channels of one tap (lanes kh = 1 hold zeros: the sums
// are those of 32 zero-padded channels, term by term).
enum Fill { C32, PAIR, SINGLE };

struct ConvArgs {
    const bf16 *in, *w;
    const float *bias;
    const bf16 *mask;
    void *out;
    const float *tg;
    double *lpart;
    int n, ntiles;
};

// Convolution on v_mfma_f32_32x32x16_bf16: rows are the 32 output channels,
// columns 32 voxels (so a lane holds four runs of four channels of one voxel
// and stores them whole).  A workgroup of 4 waves walks the tiles of X (x) by
// 2R (y) by 2 ZT (z) voxels, X = 32, 16 or 8 dividing n and R = 32 / X; a
// wave owns the X x R voxels of ZT planes.
//
// Bound by the matrix cores if they are fed: the layer's weights stay in the
// wave's registers (216 of 512 with 32 channels, so one wave per SIMD), and a
// voxel row read from LDS serves the taps of all ZT planes it touches, 0.67
// KB of LDS per instruction and wave instead of 2 KB with the weights in LDS
// as well (4 waves at 32 cycles an instruction: 85 of 128 B/cycle).  The next
// tile's halo is loaded into registers while this one is computed.  Every
// accumulator adds its taps in the order t = 0 .. 26.
// 64^3, 32 -> 32 channels: 36.8 -> 21.2 us; 5 -> 32: 17.2 -> 12.5 us; the
// 32 -> 5 layer with its loss: 41.1 + 10.8 -> 18.4 us; data gradients 52 ->
// 19.2 (5 -> 32 channels) and 21.2 us.
constexpr int kConvThreads = 256;
__host__ __device__ constexpr int fill_ch(Fill f) { return f == C32 ? 32 : 8; }
__host__ __device__ constexpr int fill_vs(Fill f) { return f == C32 ? 40 : 8; }   // LDS BF16 per voxel: 32 channels padded against bank conflicts
__host__ __device__ constexpr int fill_frags(Fill f) { return f == C32 ? 2 * kTaps : (f == PAIR ? (kTaps + 1) / 2 : kTaps); }

// Scheduling of a group of N matrix instructions: behind each one R LDS reads
// and V vector instructions, which issue while it executes.
template <int N, int R, int V> __device__ __forceinline__ void interleave()
{
    if constexpr (N > 0) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // matrix
        __builtin_amdgcn_sched_group_barrier(0x100, R, 0);   // LDS read
        __builtin_amdgcn_sched_group_barrier(0x002, V, 0);   // vector
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);   // global read
        interleave<N - 1, R, V>();
    }
}

template <Fill F, Epi E, int X, int ZT>
__global__ __launch_bounds__(kConvThreads, (F == C32 ? 1 : 2)) void k_conv(const ConvArgs A)
{
    constexpr int R = 32 / X, TY = 2 * R, TZ = 2 * ZT, HX = X + 2, HY = TY + 2, HZ = TZ + 2, HV = HX * HY * HZ;
    constexpr int CI = fill_ch(F), VS = fill_vs(F), NF = fill_frags(F), NC = CI / 8;
    constexpr int NJ = (HV * NC + kConvThreads - 1) / kConvThreads;   // halo chunks of 16 bytes per thread
    __shared__ __align__(16) bf16 sa[HV * VS];
    const int n = A.n, ntx = n / X, nty = n / TY;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wy = wave & 1, wz = wave >> 1, i = lane & 31, kh = lane >> 5;
    float bv[16];
    if constexpr (E == FWD) {
#pragma unroll
        for (int r = 0; r < 16; ++r) bv[r] = A.bias[8 * (r >> 2) + 4 * kh + (r & 3)];
    } else if constexpr (E == OUT || E == LOSS) {
#pragma unroll
        for (int r = 0; r < 4; ++r) bv[r] = A.bias && 4 * kh + r < kC3 ? A.bias[4 * kh + r] : 0.f;
    }
    double lsum = 0.0;
    int x0, y0, z0;
    auto origin = [&](int tile) {
        x0 = (tile % ntx) * X;
        tile /= ntx;
        y0 = (tile % nty) * TY;
        z0 = (tile / nty) * TZ;
    };
    // halo coordinates of the thread's chunks, the same for every tile
    int hc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int hv = min((tid + j * kConvThreads) / NC, HV - 1);
        hc[j] = hv % HX | (hv / HX % HY) << 8 | (hv / (HX * HY)) << 16;
        asm volatile("" : "+v"(hc[j]));   // keep it: the compiler would divide again for every tile
    }
    s8v pre[NJ];
    auto fetch1 = [&](int j) {   // (a thread without a last chunk loads another's again)
        const int gx = wrap(x0 - 1 + (hc[j] & 255), n), gy = wrap(y0 - 1 + (hc[j] >> 8 & 255), n),
                  gz = wrap(z0 - 1 + (hc[j] >> 16), n);
        pre[j] = *reinterpret_cast<const s8v *>(A.in + int64_t(gx + n * (gy + n * gz)) * CI + 8 * (tid % NC));
    };
    // halo voxel of the lane's voxel at tap (-1, -1, -1), plane 0 of the wave
    const bf16 *ap = sa + ((wz * ZT * HY + wy * R + i / X) * HX + i % X) * VS + (F == C32 ? 8 * kh : 0);
    constexpr auto off = [](int t) { return ((t / 9) * HY + (t / 3) % 3) * HX + t % 3; };
    const Walk walk(A.ntiles, blockIdx.x / 8, gridDim.x / 8);
    int tile = walk.first;
    origin(min(tile, A.ntiles - 1));
#pragma unroll
    for (int j = 0; j < NJ; ++j) fetch1(j);
    s8v wr[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) wr[f] = reinterpret_cast<const s8v *>(A.w)[f * 64 + lane];
    for (; tile < walk.end; tile += walk.step) {
        __syncthreads();   // the previous tile is read
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int e = tid + j * kConvThreads;
            if ((j + 1) * kConvThreads > HV * NC && e >= HV * NC) continue;
            *reinterpret_cast<s8v *>(sa + (e / NC) * VS + 8 * (e % NC)) = pre[j];
        }
        __syncthreads();
        const int gx = x0 + i % X, gy = y0 + wy * R + i / X, gz = z0 + wz * ZT;
        // the next tile's loads go between the matrix instructions (after the
        // last tile, its own again)
        origin(tile + walk.step < walk.end ? tile + walk.step : tile);
        f16v acc[ZT];
        s4v m4[ZT][4];     // MASK: the lane's mask values, LOSS: its targets, in flight meanwhile
        float tv[ZT][4];
#pragma unroll
        for (int z = 0; z < ZT; ++z) {
            const int64_t v = gx + n * (gy + n * (gz + z));   // n <= 512: 2^27 voxels
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if constexpr (E == MASK) m4[z][q] = *reinterpret_cast<const s4v *>(A.mask + v * kCP + 8 * q + 4 * kh);
                if constexpr (E == LOSS) tv[z][q] = 4 * kh + q < kC3 ? A.tg[v * kC3 + 4 * kh + q] : 0.f;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[z][r] = 0.f;
        }
        // operands are read a group ahead of the instructions that use them
        // (the compiler alone reads each just before, and a wave waits out the
        // LDS latency on every instruction)
        if constexpr (F == C32) {
            constexpr int NG = 3 * (ZT + 2);   // groups: plane p and dy, 3 dx x 2 halves of the channels
            s8v fr[2][6];
            auto read = [&](int g, s8v (&f)[6]) {
#pragma unroll
                for (int k = 0; k < 6; ++k)
                    f[k] = *reinterpret_cast<const s8v *>(ap + (g / 3 * HY * HX + g % 3 * HX + k / 2) * VS + 16 * (k % 2));
            };
            read(0, fr[0]);
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                __builtin_amdgcn_sched_barrier(0);
                if (g + 1 < NG) read(g + 1, fr[(g + 1) & 1]);
#pragma unroll
                for (int j = g * NJ / NG; j < (g + 1) * NJ / NG; ++j) fetch1(j);
                const int p = g / 3;
                int nm = 0;
#pragma unroll
                for (int k = 0; k < 6; ++k)
#pragma unroll
                    for (int z = 0; z < ZT; ++z)
                        if (p - z >= 0 && p - z < 3) {
                            acc[z] = mfma16(wr[((p - z) * 9 + g % 3 * 3) * 2 + k], fr[g & 1][k], acc[z]);
                            ++nm;
                        }
                // one LDS read and a few address instructions behind each matrix instruction
                if (nm == 12) interleave<12, 1, 4>();
                else interleave<6, 1, 7>();
            }
            __builtin_amdgcn_sched_barrier(0);
        } else {
            constexpr int GF = 4, NG = (NF + GF - 1) / GF;   // groups of 4 instructions x ZT planes
            s8v fr[2][GF * ZT];
            auto read = [&](int g, s8v (&r)[GF * ZT]) {
#pragma unroll
                for (int k = 0; k < GF; ++k) {
                    const int f = g * GF + k;
                    if (f >= NF) continue;
                    const int t0 = F == PAIR ? 2 * f : f, t1 = F == PAIR ? (2 * f + 1 < kTaps ? 2 * f + 1 : 2 * f) : f;
#pragma unroll
                    for (int z = 0; z < ZT; ++z)
                        r[k * ZT + z] = *reinterpret_cast<const s8v *>(
                            ap + ((kh ? off(t1) : off(t0)) + z * HY * HX) * VS);
                }
            };
            read(0, fr[0]);
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                __builtin_amdgcn_sched_barrier(0);
                if (g + 1 < NG) read(g + 1, fr[(g + 1) & 1]);
#pragma unroll
                for (int j = g * NJ / NG; j < (g + 1) * NJ / NG; ++j) fetch1(j);
#pragma unroll
                for (int k = 0; k < GF; ++k) {
                    const int f = g * GF + k;
                    if (f >= NF) continue;
                    const bool zero = kh && (F == SINGLE || 2 * f + 1 >= kTaps);
#pragma unroll
                    for (int z = 0; z < ZT; ++z) {
                        s8v b = fr[g & 1][k * ZT + z];
#pragma unroll
                        for (int e = 0; e < 8; ++e) b[e] = zero ? short(0) : b[e];
                        acc[z] = mfma16(wr[f], b, acc[z]);
                    }
                }
                interleave<GF * ZT, 1, 7>();
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int z = 0; z < ZT; ++z) {
            const int64_t v = gx + n * (gy + n * (gz + z));
            if constexpr (E == FWD || E == MASK) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float x[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        float val = acc[z][4 * q + k];
                        if constexpr (E == FWD) {
                            val += bv[4 * q + k];
                            x[k] = val > 0.f ? val : 0.f;
                        } else {
                            x[k] = from_bf16(bf16(m4[z][q][k])) > 0.f ? val : 0.f;
                        }
                    }
                    *reinterpret_cast<s4v *>(static_cast<bf16 *>(A.out) + v * kCP + 8 * q + 4 * kh) = pack4(x);
                }
            } else if constexpr (E == OUT) {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (4 * kh + k < kC3) {
                        float val = acc[z][k];
                        if (A.bias) val += bv[k];
                        static_cast<float *>(A.out)[v * kC3 + 4 * kh + k] = val;
                    }
            } else {
                const float sc = 2.0f / (5.0f * (float(n) * float(n) * float(n)));
                float x[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    float gv = 0.f;
                    if (4 * kh + k < kC3) {
                        float val = acc[z][k];
                        val += bv[k];
                        const float d = val - tv[z][k];
                        lsum += double(d) * double(d);
                        gv = sc * d;
                    }
                    x[k] = gv;
                }
                if (A.out) *reinterpret_cast<s4v *>(static_cast<bf16 *>(A.out) + v * kC0P + 4 * kh) = pack4(x);
            }
        }
    }
    if constexpr (E == LOSS) {
        __shared__ double wl[4];
        for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o);
        if (lane == 0) wl[wave] = lsum;
        __syncthreads();
        if (tid == 0) A.lpart[blockIdx.x] = ((wl[0] + wl[1]) + wl[2]) + wl[3];
    }
}

// Tiles of a convolution: 256 voxels, or 128 where 256-voxel ones would be
// fewer than two per CU (32^3 has 128 of them for 256 CUs).
struct ConvGrid { int zt, ntiles, blocks; };
constexpr int kConvBlocks = 256;   // persistent workgroups (CUs) of a convolution, at most
__host__ inline ConvGrid conv_grid(int n)
{
    const int64_t v = int64_t(n) * n * n;
    ConvGrid g;
    g.zt = v / 256 >= 2 * kConvBlocks ? 2 : 1;
    g.ntiles = int(v / (128 * g.zt));
    g.blocks = 8 * std::min((g.ntiles + 7) / 8, kConvBlocks / 8);
    return g;
}

// Weight and bias gradients of a layer as a GEMM over voxels:
// gW[o][t][c] = sum_v go[v][o] act[nb(v, t)][c] and gb[o] = sum_v go[v][o].
// Slot b of G = min(V / 256, 256) takes the 256-voxel tiles b, b + G, ... (X
// by 2R by 4 voxels, as the convolutions') and one workgroup; each gradient
// entry of a slot is one chain of matrix instructions over its tiles' 16-voxel
// runs in order, and k_grad_slices and k_grad_adam add the slots in order (no
// atomics).  Training amplifies a last-bit change of a gradient to 1e-4 of the
// parameters within 40 iterations, so this order is part of the result.
//
// Both operands come from channel-last rows: the gfx950 transposing LDS read
// gives lane l of 16 the l-th of the 16 channels its group reads for four
// voxels, so two of them make an operand's eight voxels per lane (before:
// eight 2-byte reads per operand).  The next tile's loads go between the
// matrix instructions.
constexpr int kWgThreads = 512, kWgSlots = 256;
__host__ inline int wg_slots(int n)
{
    const int64_t tiles = int64_t(n) * n * n / 256;
    return tiles < kWgSlots ? int(tiles) : kWgSlots;
}
// the slot of a workgroup: neighbouring slots on one XCD where they divide evenly
__device__ __forceinline__ int wg_slot()
{
    const int G = gridDim.x;
    return G % 8 == 0 ? int(blockIdx.x % 8) * (G / 8) + int(blockIdx.x / 8) : int(blockIdx.x);
}

__device__ __forceinline__ s8v tr_read(const bf16 *lo, const bf16 *hi)
{
    const s4v a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(lo)),
              b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(hi));
    s8v r;
#pragma unroll
    for (int k = 0; k < 4; ++k) { r[k] = a[k]; r[4 + k] = b[k]; }
    return r;
}

// A tile's halo of CA-channel activations and its GC-channel output gradient,
// staged through registers: NJ 16-byte chunks per thread.
template <int X, int CA, int GC> struct WgTile {
    static constexpr int R = 32 / X, TY = 2 * R, HX = X + 2, HY = TY + 2, HV = HX * HY * 6;
    static constexpr int NCA = CA / 8, NCG = GC / 8, NA = HV * NCA, NG = 256 * NCG;
    static constexpr int JA = (NA + kWgThreads - 1) / kWgThreads, JG = (NG + kWgThreads - 1) / kWgThreads, NJ = JA + JG;
    // a lane's first voxel of run q = 4 lz + qq sits at its base + row(qq) + lz planes
    static constexpr int row(int qq) { return X == 32 ? (qq >> 1) * HX + 16 * (qq & 1) : (X == 16 ? qq * HX : 2 * qq * HX); }
    static constexpr int half_step() { return X == 8 ? HX : 8; }   // to the second eight voxels of a run
    int x0, y0, z0, n;
    const bf16 *act, *go;
    __device__ void origin(int tile)
    {
        const int ntx = n / X, nty = n / TY;
        x0 = (tile % ntx) * X;
        y0 = (tile / ntx % nty) * TY;
        z0 = tile / (ntx * nty) * 4;
    }
    __device__ __forceinline__ s8v fetch(int j) const   // (a thread without a last chunk loads another's again)
    {
        const int tid = threadIdx.x;
        if (j < JA) {
            const int hv = min((tid + j * kWgThreads) / NCA, HV - 1);
            const int gx = wrap(x0 - 1 + hv % HX, n), gy = wrap(y0 - 1 + hv / HX % HY, n),
                      gz = wrap(z0 - 1 + hv / (HX * HY), n);
            return *reinterpret_cast<const s8v *>(act + int64_t(gx + n * (gy + n * gz)) * CA + 8 * (tid % NCA));
        }
        const int vl = min((tid + (j - JA) * kWgThreads) / NCG, 255);
        const int v = x0 + vl % X + n * (y0 + vl / X % TY + n * (z0 + vl / (X * TY)));
        return *reinterpret_cast<const s8v *>(go + int64_t(v) * GC + 8 * (tid % NCG));
    }
    __device__ __forceinline__ void put(int j, const s8v &x, bf16 *sa, bf16 *sg) const
    {
        const int e = threadIdx.x + (j < JA ? j : j - JA) * kWgThreads;
        if (j < JA) {
            if ((j + 1) * kWgThreads <= NA || e < NA) *reinterpret_cast<s8v *>(sa + 8 * e) = x;
        } else if ((j - JA + 1) * kWgThreads <= NG || e < NG) {
            *reinterpret_cast<s8v *>(sg + 8 * e) = x;
        }
    }
};

// LDS of the kernels below (BF16 values): halo, output gradient and, for 8 of
// them, as many zeros for the absent channels
template <int X, int CA, int GC> constexpr size_t wg_lds()
{
    return sizeof(bf16) * (size_t(WgTile<X, CA, GC>::HV) * CA + 256 * GC * (GC == 8 ? 2 : 1));
}

// Against 32-channel activations (layers 2 and 3; the latter with the 8-channel
// output gradient).  Wave w < 8 owns the taps of (dy, dx) = (w / 3, w % 3) for
// the three dz, so a row of activations read once serves three instructions;
// the three taps left, (dy, dx) = (2, 2), go to waves 0 to 2: 13 or 14 taps on
// each SIMD.  64^3: 55 -> 20.5 (layer 2) and 16.4 us (layer 3).
template <int X, int GC>
__global__ __launch_bounds__(kWgThreads, 2) void k_wgrad32(const bf16 *__restrict__ go, const bf16 *__restrict__ act,
                                                           float *__restrict__ part, float *__restrict__ bpart, int n,
                                                           int ntiles)
{
    using T = WgTile<X, kCP, GC>;
    constexpr int P = T::HY * T::HX;
    extern __shared__ __align__(16) unsigned short wg_mem[];
    bf16 *sa = wg_mem, *sg = wg_mem + T::HV * kCP;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, kh = lane >> 5;
    const int lv = (lane & 15) >> 2, lc = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);   // voxel and channel the lane loads
    if constexpr (GC == 8)
        for (int e = tid; e < 256 * GC; e += kWgThreads) sg[256 * GC + e] = 0;
    const bf16 *gp = sg + (GC == 8 && lc >= GC ? 256 * GC : (8 * kh + lv) * GC + lc);
    const int lane_at = (lv + kh * T::half_step()) * kCP + lc;
    const bf16 *bp = sa + ((wave / 3) * T::HX + wave % 3) * kCP + lane_at;
    const bf16 *bx = sa + ((min(wave, 2)) * P + 2 * T::HX + 2) * kCP + lane_at;
    f16v acc[3], accx;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = acc[2][r] = accx[r] = 0.f;
    float bsum = 0.f;
    T t;
    t.n = n;
    t.act = act;
    t.go = go;
    const int slot = wg_slot();
    t.origin(slot);
    s8v pre[T::NJ];
#pragma unroll
    for (int j = 0; j < T::NJ; ++j) pre[j] = t.fetch(j);
    for (int tile = slot; tile < ntiles; tile += gridDim.x) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < T::NJ; ++j) t.put(j, pre[j], sa, sg);
        __syncthreads();
        t.origin(tile + int(gridDim.x) < ntiles ? tile + int(gridDim.x) : tile);
        s8v g[16], br[2][4];
        auto read_g = [&](int lz) {
#pragma unroll
            for (int qq = 0; qq < 4; ++qq) {
                const bf16 *q = gp + 16 * (4 * lz + qq) * GC;
                g[4 * lz + qq] = tr_read(q, q + 4 * GC);
            }
        };
        auto read_b = [&](int p, const bf16 *base, s8v (&b)[4]) {
#pragma unroll
            for (int qq = 0; qq < 4; ++qq) {
                const bf16 *q = base + (p * P + T::row(qq)) * kCP;
                b[qq] = tr_read(q, q + 4 * kCP);
            }
        };
        read_g(0);
        read_b(0, bp, br[0]);
#pragma unroll
        for (int p = 0; p < 6; ++p) {
            __builtin_amdgcn_sched_barrier(0);
            if (p + 1 < 4) read_g(p + 1);
            if (p + 1 < 6) read_b(p + 1, bp, br[(p + 1) & 1]);
#pragma unroll
            for (int j = p * T::NJ / 6; j < (p + 1) * T::NJ / 6; ++j) pre[j] = t.fetch(j);
#pragma unroll
            for (int dz = 0; dz < 3; ++dz)
                if (p - dz >= 0 && p - dz < 4) {
#pragma unroll
                    for (int qq = 0; qq < 4; ++qq) acc[dz] = mfma16(g[4 * (p - dz) + qq], br[p & 1][qq], acc[dz]);
                }
            if (p == 0 || p == 5) interleave<4, 4, 10>();
            else if (p == 1 || p == 4) interleave<8, 2, 6>();
            else interleave<12, 2, 4>();
        }
        __builtin_amdgcn_sched_barrier(0);
        if (wave < 3) {
            read_b(0, bx, br[0]);
#pragma unroll
            for (int lz = 0; lz < 4; ++lz) {
                __builtin_amdgcn_sched_barrier(0);
                if (lz < 3) read_b(lz + 1, bx, br[(lz + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int qq = 0; qq < 4; ++qq) accx = mfma16(g[4 * lz + qq], br[lz & 1][qq], accx);
            }
        } else if (wave == 7) {
#pragma unroll
            for (int q = 0; q < 16; ++q)
#pragma unroll
                for (int e = 0; e < 8; ++e) bsum += from_bf16(bf16(g[q][e]));
        }
    }
    auto store = [&](int tap, const f16v &a) {
#pragma unroll
        for (int q = 0; q < GC / 8; ++q) {
            f4v x;
#pragma unroll
            for (int k = 0; k < 4; ++k) x[k] = a[4 * q + k];
            *reinterpret_cast<f4v *>(part + ((int64_t(slot) * kTaps + tap) * (GC / 8) + q) * 256 + 4 * lane) = x;
        }
    };
#pragma unroll
    for (int dz = 0; dz < 3; ++dz) store(9 * dz + wave, acc[dz]);
    if (wave < 3) store(9 * wave + 8, accx);
    if (wave == 7) {
        bsum += __shfl_xor(bsum, 32);
        if (lane < kCP) bpart[slot * kCP + lane] = bsum;
    }
}

// Against the 8-channel input (layer 1): the 27 x 8 columns in seven tiles of
// four taps, one per wave; wave 7 sums the bias.  64^3: 26.7 -> 10.3 us.
template <int X>
__global__ __launch_bounds__(kWgThreads, 2) void k_wgrad8(const bf16 *__restrict__ go, const bf16 *__restrict__ act,
                                                          float *__restrict__ part, float *__restrict__ bpart, int n,
                                                          int ntiles)
{
    using T = WgTile<X, kC0P, kCP>;
    constexpr int P = T::HY * T::HX;
    extern __shared__ __align__(16) unsigned short wg_mem[];
    bf16 *sa = wg_mem, *sg = wg_mem + T::HV * kC0P;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, kh = lane >> 5;
    const int lv = (lane & 15) >> 2, half = (lane >> 4) & 1;
    const bf16 *gp = sg + (8 * kh + lv) * kCP + 16 * half + 4 * (lane & 3);
    // the lane loads 4 channels of tap 4 wave + 2 half + ((lane & 3) >> 1);
    // the columns of a 28th tap (and wave 7's) are never read
    const int tap = min(4 * wave + 2 * half + ((lane & 3) >> 1), kTaps - 1);
    const bf16 *bp = sa + (tap / 9 * P + tap / 3 % 3 * T::HX + tap % 3 + lv + kh * T::half_step()) * kC0P + 4 * (lane & 1);
    f16v acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    float bsum = 0.f;
    T t;
    t.n = n;
    t.act = act;
    t.go = go;
    const int slot = wg_slot();
    t.origin(slot);
    s8v pre[T::NJ];
#pragma unroll
    for (int j = 0; j < T::NJ; ++j) pre[j] = t.fetch(j);
    for (int tile = slot; tile < ntiles; tile += gridDim.x) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < T::NJ; ++j) t.put(j, pre[j], sa, sg);
        __syncthreads();
        t.origin(tile + int(gridDim.x) < ntiles ? tile + int(gridDim.x) : tile);
        s8v g[2][4], br[2][4];
        auto read = [&](int lz) {
#pragma unroll
            for (int qq = 0; qq < 4; ++qq) {
                const bf16 *q = gp + 16 * (4 * lz + qq) * kCP, *b = bp + (lz * P + T::row(qq)) * kC0P;
                g[lz & 1][qq] = tr_read(q, q + 4 * kCP);
                br[lz & 1][qq] = tr_read(b, b + 4 * kC0P);
            }
        };
        read(0);
#pragma unroll
        for (int lz = 0; lz < 4; ++lz) {
            __builtin_amdgcn_sched_barrier(0);
            if (lz < 3) read(lz + 1);
#pragma unroll
            for (int j = lz * T::NJ / 4; j < (lz + 1) * T::NJ / 4; ++j) pre[j] = t.fetch(j);
            if (wave == 7) {
#pragma unroll
                for (int qq = 0; qq < 4; ++qq)
#pragma unroll
                    for (int e = 0; e < 8; ++e) bsum += from_bf16(bf16(g[lz & 1][qq][e]));
            } else {
#pragma unroll
                for (int qq = 0; qq < 4; ++qq) acc = mfma16(g[lz & 1][qq], br[lz & 1][qq], acc);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if (wave < 7) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            f4v x;
#pragma unroll
            for (int k = 0; k < 4; ++k) x[k] = acc[4 * q + k];
            *reinterpret_cast<f4v *>(part + ((int64_t(slot) * 7 + wave) * 4 + q) * 256 + 4 * lane) = x;
        }
    } else {
        bsum += __shfl_xor(bsum, 32);
        if (lane < kCP) bpart[slot * kCP + lane] = bsum;
    }
}

// First level of the gradient reductions, all layers in one launch: out[s][k]
// = sum over slice s of the G slots of element k of a slice (kS2, kS1, ...):
// slots s per .. in order for the weights, s, s + 8, ... for the biases.
struct GradParts { const float *p2, *p1, *p3, *b1, *b2, *b3; };
__global__ __launch_bounds__(256) void k_grad_slices(const GradParts P, float *__restrict__ out, int G)
{
    const int k = blockIdx.x * 256 + threadIdx.x, sl = blockIdx.y;
    if (k >= kSlice) return;
    const float *src;
    int stride, c0, c1, step;
    if (k < kSB1) {
        if (k < kS1) { src = P.p2 + k; stride = kP2; }
        else if (k < kS3) { src = P.p1 + (k - kS1); stride = kP1; }
        else { src = P.p3 + (k - kS3); stride = kP3; }
        const int per = (G + kWgSlices - 1) / kWgSlices;
        c0 = sl * per;
        c1 = min(G, c0 + per);
        step = 1;
    } else {
        src = k < kSB2 ? P.b1 + (k - kSB1) : (k < kSB3 ? P.b2 + (k - kSB2) : P.b3 + (k - kSB3));
        stride = kCP;
        c0 = sl;
        c1 = G;
        step = kWgSlices;
    }
    float s = 0.f;
#pragma unroll 8
    for (int c = c0; c < c1; c += step) s += src[int64_t(c) * stride];
    out[int64_t(sl) * kSlice + k] = s;
}

// loss += the sum of lpart[0 .. nb - 1] (one workgroup of 256, slices summed
// in order).
__device__ __forceinline__ void loss_add(const double *__restrict__ lpart, double *__restrict__ loss, int nb)
{
    __shared__ double sl[256];
    double s = 0.0;
    for (int b = threadIdx.x; b < nb; b += 256) s += lpart[b];
    sl[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (int(threadIdx.x) < w) sl[threadIdx.x] += sl[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *loss += sl[0];
}
__global__ __launch_bounds__(256) void k_loss_add(const double *__restrict__ lpart, double *__restrict__ loss, int nb)
{
    loss_add(lpart, loss, nb);
}

// BF16 [V][8] from FP32 [V][5] (inputs and output gradients of the test hooks).
__global__ void k_pack_host_in(const float *__restrict__ x, bf16 *__restrict__ a, int V)
{
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v >= V) return;
    for (int c = 0; c < kC0P; ++c) a[int64_t(v) * kC0P + c] = to_bf16(c < kC0 ? x[int64_t(v) * kC0 + c] : 0.f);
}

struct Norm {
    float in_mean[5], in_scale[5], out_scale[5];
};

// Normalised network input from the state of a block with n+1 stored points
// per direction (unique points 0..n-1).
__global__ void k_pack_state(const double *__restrict__ q, int64_t NT, int64_t off, int n, Norm nm,
                             bf16 *__restrict__ a)
{
    const int V = n * n * n;
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v >= V) return;
    const int x = v % n, y = (v / n) % n, z = v / (n * n);
    const int64_t g = off + x + int64_t(n + 1) * (y + int64_t(n + 1) * z);
    for (int c = 0; c < kC0P; ++c) {
        float f = 0.f;
        if (c < kC0) f = float((q[c * NT + g] - double(nm.in_mean[c])) / double(nm.in_scale[c]));
        a[int64_t(v) * kC0P + c] = to_bf16(f);
    }
}

// q += correction (denormalised) at every stored point of the block.
__global__ void k_add_correction(double *__restrict__ q, int64_t NT, int64_t off, int n, Norm nm,
                                 const float *__restrict__ y)
{
    const int np = n + 1;
    const int64_t P = int64_t(np) * np * np;
    const int64_t l = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (l >= P) return;
    const int x = int(l % np), yy = int((l / np) % np), z = int(l / (int64_t(np) * np));
    const int64_t v = (x % n) + int64_t(n) * ((yy % n) + int64_t(n) * (z % n));
    for (int c = 0; c < kC3; ++c) q[c * NT + off + l] += double(y[v * kC3 + c]) * double(nm.out_scale[c]);
}

// Top-hat filter of width r fine cells (trapezoidal weights 1/2, 1, .., 1,
// 1/2 over r+1 points, divided by r per direction) of a periodic fine block
// (nf+1 points per direction) sampled at the coarse points, into a coarse
// block with n+1 points per direction; nf = r n.
__global__ void k_box(const double *__restrict__ qf, int64_t NTf, int64_t offf, int nf, double *__restrict__ qc,
                      int64_t NTc, int64_t offc, int n, int r)
{
    const int np = n + 1, nfp = nf + 1;
    const int64_t P = int64_t(np) * np * np;
    const int64_t l = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (l >= P) return;
    const int x = int(l % np), y = int((l / np) % np), z = int(l / (int64_t(np) * np));
    const int h = r / 2;
    double s[5] = {0, 0, 0, 0, 0};
    for (int c = -h; c <= h; ++c) {
        const double wc = (c == -h || c == h) ? 0.5 : 1.0;
        const int fz = ((z * r + c) % nf + nf) % nf;
        for (int b = -h; b <= h; ++b) {
            const double wb = wc * ((b == -h || b == h) ? 0.5 : 1.0);
            const int fy = ((y * r + b) % nf + nf) % nf;
            for (int a = -h; a <= h; ++a) {
                const double w = wb * ((a == -h || a == h) ? 0.5 : 1.0);
                const int fx = ((x * r + a) % nf + nf) % nf;
                const int64_t g = offf + fx + int64_t(nfp) * (fy + int64_t(nfp) * fz);
                for (int m = 0; m < 5; ++m) s[m] += w * qf[m * NTf + g];
            }
        }
    }
    const double inv = 1.0 / (double(r) * r * r);
    for (int m = 0; m < 5; ++m) qc[m * NTc + offc + l] = s[m] * inv;
}

// Training pair: input = packed coarse state, target = (filtered fine - coarse) / out_scale.
__global__ void k_target(const double *__restrict__ qc, int64_t NTc, int64_t offc, const double *__restrict__ qt,
                         int64_t NTt, int64_t offt, int n, Norm nm, float *__restrict__ tg)
{
    const int V = n * n * n;
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v >= V) return;
    const int x = v % n, y = (v / n) % n, z = v / (n * n);
    const int64_t l = x + int64_t(n + 1) * (y + int64_t(n + 1) * z);
    for (int c = 0; c < kC3; ++c)
        tg[int64_t(v) * kC3 + c] =
            float((qt[c * NTt + offt + l] - qc[c * NTc + offc + l]) / double(nm.out_scale[c]));
}

// BF16 weights as the convolutions' lanes hold them: [instruction][lane][8],
// lane = 32 (K half) + row.  wf1 (PAIR), wf2, wf3 (C32): forward, rows are
// output channels; wd3 (SINGLE), wd2, wd1 (C32): data gradients, rows are
// input channels and the tap is the opposite one.  Rows and channels without
// a parameter stay zero.
struct Wts {
    bf16 *wf1, *wf2, *wf3, *wd1, *wd2, *wd3;
};
constexpr int64_t frag_size(Fill f) { return int64_t(fill_frags(f)) * 64 * 8; }

__device__ __forceinline__ int frag_c32(int t, int ch, int row)
{
    return (((2 * t + (ch >> 4)) * 64) + ((ch >> 3) & 1) * 32 + row) * 8 + (ch & 7);
}
// Parameter k (value x) into the layouts it appears in.
__device__ __forceinline__ void put_weight(const Wts &W, int k, float x)
{
    const bf16 h = to_bf16(x);
    if (k < kOB1) {
        const int o = k / (kTaps * kC0), t = k / kC0 % kTaps, c = k % kC0;
        W.wf1[((t >> 1) * 64 + (t & 1) * 32 + o) * 8 + c] = h;
        W.wd1[frag_c32(kTaps - 1 - t, o, c)] = h;
    } else if (k >= kOW2 && k < kOB2) {
        const int e = k - kOW2, o = e / (kTaps * kC1), t = e / kC1 % kTaps, c = e % kC1;
        W.wf2[frag_c32(t, c, o)] = h;
        W.wd2[frag_c32(kTaps - 1 - t, o, c)] = h;
    } else if (k >= kOW3 && k < kOB3) {
        const int e = k - kOW3, o = e / (kTaps * kC2), t = e / kC2 % kTaps, c = e % kC2;
        W.wf3[frag_c32(t, c, o)] = h;
        W.wd3[((kTaps - 1 - t) * 64 + c) * 8 + o] = h;
    }
}
__global__ __launch_bounds__(256) void k_prep(const float *__restrict__ p, Wts W)
{
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k < kNParam) put_weight(W, k, p[k]);
}

// Place of parameter k in a slice: row r and column m of an accumulator tile
// sit at lane 32 ((r >> 2) & 1) + m, value 4 (r >> 3) + r % 4.
__device__ __forceinline__ int slice_at(int r, int m)
{
    return ((r >> 3) * 64 + ((r >> 2) & 1) * 32 + m) * 4 + (r & 3);
}
__device__ __forceinline__ int slice_index(int k)
{
    if (k < kOB1) {
        const int o = k / (kTaps * kC0), m = (k / kC0 % kTaps) * kC0P + k % kC0;
        return kS1 + (m >> 5) * 1024 + slice_at(o, m & 31);
    }
    if (k < kOW2) return kSB1 + k - kOB1;
    if (k < kOB2) {
        const int e = k - kOW2;
        return kS2 + e / kC1 % kTaps * 1024 + slice_at(e / (kTaps * kC1), e % kC1);
    }
    if (k < kOW3) return kSB2 + k - kOB2;
    if (k < kOB3) {
        const int e = k - kOW3;
        return kS3 + e / kC2 % kTaps * 256 + slice_at(e / (kTaps * kC2), e % kC2);
    }
    return kSB3 + k - kOB3;
}

// Second level: the flat gradient g from the slices and, with update, the
// Adam update of the parameters and their BF16 copies; the last workgroup
// adds the nl partial losses to the running loss (lpart null: no loss).
__global__ __launch_bounds__(256) void k_grad_adam(const float *__restrict__ slices, float *__restrict__ g,
                                                   float *__restrict__ p, float *__restrict__ m1,
                                                   float *__restrict__ m2, Wts W, int update, float lr, float c1,
                                                   float c2,
                                                   const double *__restrict__ lpart, double *__restrict__ loss, int nl)
{
    if (blockIdx.x == gridDim.x - 1) {
        if (lpart) loss_add(lpart, loss, nl);
        return;
    }
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= kNParam) return;
    const int at = slice_index(k);
    float gk = 0.f;
#pragma unroll
    for (int s = 0; s < kWgSlices; ++s) gk += slices[s * kSlice + at];
    g[k] = gk;
    if (!update) return;
    constexpr float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float a = b1 * m1[k] + (1.f - b1) * gk, b = b2 * m2[k] + (1.f - b2) * gk * gk;
    m1[k] = a;
    m2[k] = b;
    const float x = p[k] - lr * (a / c1) / (sqrtf(b / c2) + eps);
    p[k] = x;
    put_weight(W, k, x);
}

__global__ void k_fill(float *a, float v, int64_t n)
{
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) a[i] = v;
}

}  // namespace

// Device scratch of cnd_net_apply_noalloc: the network input, the two
// hidden activations and the output of one apply on an n^3 grid with n up
// to kScratchN (V = n^3 voxels: BF16 [V][8], [V][32], [V][32], FP32 [V][5],
// each part aligned to 256 bytes), 41 MiB.  Every GPU the library runs on
// holds its own copy until the process ends; host code reaches it only
// through the address hipGetSymbolAddress gives for the current device.
constexpr int kScratchN = 64;
constexpr size_t kScratchV = size_t(kScratchN) * kScratchN * kScratchN;
constexpr size_t align256(size_t b) { return (b + 255) / 256 * 256; }
constexpr size_t kScratchBytes = align256(kScratchV * 8 * 2) + 2 * align256(kScratchV * 32 * 2) +
                                 align256(kScratchV * 5 * 4);
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

struct cnd_net {
    int n = 0, V = 0, cap = 0, npairs = 0;
    hipStream_t st = nullptr;
    // recorded after every use of the network's activation buffers, on
    // whichever stream ran it; the next use waits for it first, so calls on
    // different streams (one per context) never overlap on those buffers
    hipEvent_t done = nullptr;
    Norm nm{};
    float *p = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;   // parameters, gradient, Adam moments
    // weight and bias gradients per workgroup (layers 2, 1 and 3), and per
    // slice of workgroups
    float *gp2 = nullptr, *gp1 = nullptr, *gp3 = nullptr, *b1 = nullptr, *b2 = nullptr, *b3 = nullptr;
    float *slices = nullptr;
    Wts W{};
    bf16 *x0 = nullptr, *a1 = nullptr, *a2 = nullptr, *g3 = nullptr, *g2 = nullptr, *g1 = nullptr;
    float *y = nullptr, *gx = nullptr, *hx = nullptr;
    double *loss = nullptr, *lpart = nullptr;   // running loss, per-workgroup sums of one pair
    bf16 *din = nullptr;    // pairs: inputs [cap][V][8]
    float *dtg = nullptr;   // pairs: targets [cap][V][5]
    long long adam_t = 0;
    std::string err;
};

namespace {

thread_local std::string g_net_err;

int nfail(cnd_net *net, int code, const std::string &m)
{
    if (net) net->err = m; else g_net_err = m;
    return code;
}

#define NHIP(net, call)                                                                             \
    do {                                                                                            \
        hipError_t e_ = (call);                                                                     \
        if (e_ != hipSuccess) return nfail((net), CND_EDEVICE, std::string(#call ": ") + hipGetErrorString(e_)); \
    } while (0)

inline unsigned blocks_for(int64_t n, int per) { return unsigned((n + per - 1) / per); }

int net_begin(cnd_net *t, hipStream_t st);
int net_end(cnd_net *t, hipStream_t st);

int prep(cnd_net *t, hipStream_t st)
{
    hipLaunchKernelGGL(k_prep, dim3(blocks_for(kNParam, 256)), dim3(256), 0, st, t->p, t->W);
    NHIP(t, hipGetLastError());
    return CND_OK;
}

template <Fill F, Epi E>
void conv(cnd_net *t, hipStream_t st, const bf16 *in, const bf16 *w, const float *bias, const bf16 *mask, void *out,
          const float *tg = nullptr)
{
    const ConvGrid g = conv_grid(t->n);
    const ConvArgs A{in, w, bias, mask, out, tg, t->lpart, t->n, g.ntiles};
    const dim3 gr(unsigned(g.blocks)), b(kConvThreads);
    auto go = [&](auto x) {
        constexpr int X = decltype(x)::value;
        if (g.zt == 2) hipLaunchKernelGGL((k_conv<F, E, X, 2>), gr, b, 0, st, A);
        else hipLaunchKernelGGL((k_conv<F, E, X, 1>), gr, b, 0, st, A);
    };
    const int x = conv_x(t->n);
    if (x == 32) go(std::integral_constant<int, 32>{});
    else if (x == 16) go(std::integral_constant<int, 16>{});
    else go(std::integral_constant<int, 8>{});
}

// the hidden activations a1, a2 (BF16 [V][32]) of the input x0
void hidden(cnd_net *t, const bf16 *x0, bf16 *a1, bf16 *a2, hipStream_t st)
{
    conv<PAIR, FWD>(t, st, x0, t->W.wf1, t->p + kOB1, nullptr, a1);
    conv<C32, FWD>(t, st, a1, t->W.wf2, t->p + kOB2, nullptr, a2);
}

// forward of the input in x0 into y (normalised correction, FP32 [V][5])
int forward_into(cnd_net *t, const bf16 *x0, bf16 *a1, bf16 *a2, float *y, hipStream_t st)
{
    hidden(t, x0, a1, a2, st);
    conv<C32, OUT>(t, st, a2, t->W.wf3, t->p + kOB3, nullptr, y);
    NHIP(t, hipGetLastError());
    return CND_OK;
}

// ... with the network's own buffers
int forward(cnd_net *t, const bf16 *x0, hipStream_t st) { return forward_into(t, x0, t->a1, t->a2, t->y, st); }

// q += correction(q) on the coarse block C with the buffers x0, a1, a2, y
// (cnd_net_apply and its variant without allocations)
int apply_into(cnd_net *t, const CtxView &C, bf16 *x0, bf16 *a1, bf16 *a2, float *y)
{
    int r;
    if ((r = net_begin(t, C.st))) return r;
    const int64_t V = t->V;
    hipLaunchKernelGGL(k_pack_state, dim3(blocks_for(V, 256)), dim3(256), 0, C.st, C.q, C.NT, C.off, t->n, t->nm, x0);
    if ((r = forward_into(t, x0, a1, a2, y, C.st))) return r;
    const int64_t P = int64_t(t->n + 1) * (t->n + 1) * (t->n + 1);
    hipLaunchKernelGGL(k_add_correction, dim3(blocks_for(P, 256)), dim3(256), 0, C.st, C.q, C.NT, C.off, t->n, t->nm,
                       y);
    return net_end(t, C.st);
}

// Sums of the squared errors of the pair (x0, tg) into lpart and, with g3,
// the loss gradient.
void forward_loss(cnd_net *t, const bf16 *x0, const float *tg, bf16 *g3, hipStream_t st)
{
    hidden(t, x0, t->a1, t->a2, st);
    conv<C32, LOSS>(t, st, t->a2, t->W.wf3, t->p + kOB3, nullptr, g3, tg);
}

// Weight and bias gradients of layer 1, 2 or 3 from its output gradient go and
// its input act.
void wgrad(cnd_net *t, hipStream_t st, int layer, const bf16 *go, const bf16 *act, float *part, float *bpart)
{
    const int tiles = t->V / 256;
    const dim3 g(unsigned(wg_slots(t->n))), b(kWgThreads);
    auto run = [&](auto x) {
        constexpr int X = decltype(x)::value;
        if (layer == 1)
            hipLaunchKernelGGL(k_wgrad8<X>, g, b, (wg_lds<X, kC0P, kCP>()), st, go, act, part, bpart, t->n, tiles);
        else if (layer == 2)
            hipLaunchKernelGGL((k_wgrad32<X, kCP>), g, b, (wg_lds<X, kCP, kCP>()), st, go, act, part, bpart, t->n, tiles);
        else
            hipLaunchKernelGGL((k_wgrad32<X, kC0P>), g, b, (wg_lds<X, kCP, kC0P>()), st, go, act, part, bpart, t->n,
                               tiles);
    };
    const int x = conv_x(t->n);
    if (x == 32) run(std::integral_constant<int, 32>{});
    else if (x == 16) run(std::integral_constant<int, 16>{});
    else run(std::integral_constant<int, 8>{});
}

// backward from g3 (dL/dy, BF16 [V][8]) with the activations of the last
// forward: slices of the parameter gradient; with gx, dL/dx0 into gx (FP32
// [V][5]).
int backward(cnd_net *t, const bf16 *x0, float *gx, hipStream_t st)
{
    wgrad(t, st, 3, t->g3, t->a2, t->gp3, t->b3);
    conv<SINGLE, MASK>(t, st, t->g3, t->W.wd3, nullptr, t->a2, t->g2);
    wgrad(t, st, 2, t->g2, t->a1, t->gp2, t->b2);
    conv<C32, MASK>(t, st, t->g2, t->W.wd2, nullptr, t->a1, t->g1);
    wgrad(t, st, 1, t->g1, x0, t->gp1, t->b1);
    if (gx) conv<C32, OUT>(t, st, t->g1, t->W.wd1, nullptr, nullptr, gx);
    hipLaunchKernelGGL(k_grad_slices, dim3(blocks_for(kSlice, 256), kWgSlices), dim3(256), 0, st,
                       GradParts{t->gp2, t->gp1, t->gp3, t->b1, t->b2, t->b3}, t->slices, wg_slots(t->n));
    NHIP(t, hipGetLastError());
    return CND_OK;
}

// The flat gradient from the slices and, with update, the Adam step; with nl,
// the partial losses of the pair to the running loss.
void finish(cnd_net *t, bool update, float lr, float c1, float c2, int nl, hipStream_t st)
{
    hipLaunchKernelGGL(k_grad_adam, dim3(blocks_for(kNParam, 256) + 1), dim3(256), 0, st, t->slices, t->g, t->p, t->m1,
                       t->m2, t->W, update ? 1 : 0, lr, c1, c2, nl ? t->lpart : nullptr, t->loss, nl);
}

template <class T>
int nalloc(cnd_net *t, T **p, int64_t n)
{
    NHIP(t, hipMalloc((void **)p, size_t(std::max<int64_t>(n, 1)) * sizeof(T)));
    return CND_OK;
}

// Order work on st after every earlier use of the network's buffers, and
// mark the end of this use.
int net_begin(cnd_net *t, hipStream_t st)
{
    NHIP(t, hipStreamWaitEvent(st, t->done, 0));
    return CND_OK;
}
int net_end(cnd_net *t, hipStream_t st)
{
    NHIP(t, hipGetLastError());
    NHIP(t, hipEventRecord(t->done, st));
    return CND_OK;
}

// The address of scratch on the current device, looked up once per device
// (the first call on it) and kept; nullptr and the error if that fails.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch[kMaxDevices] = {};

void *scratch_address(cnd_net *t)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        nfail(t, CND_EDEVICE, "cnd_net_apply_noalloc: no current device");
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            nfail(t, CND_EDEVICE, std::string("cnd_net_apply_noalloc: hipGetSymbolAddress: ") + hipGetErrorString(e));
            return nullptr;
        }
        g_scratch[dev] = ptr;
    }
    return g_scratch[dev];
}

}  // namespace

extern "C" {

int cnd_net_param_count(void) { return kNParam; }

const char *cnd_net_error(const cnd_net *net) { return net ? net->err.c_str() : g_net_err.c_str(); }

int cnd_net_create(int n, int capacity, unsigned long long seed, cnd_net **out)
{
    if (!out) return nfail(nullptr, CND_EINVAL, "cnd_net_create: null output");
    *out = nullptr;
    if (n < 8 || n % 8 != 0 || n > 512) return nfail(nullptr, CND_EINVAL, "cnd_net_create: n must be a multiple of 8 in 8..512");
    if (capacity < 0) return nfail(nullptr, CND_EINVAL, "cnd_net_create: negative capacity");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return nfail(nullptr, CND_EDEVICE, "no HIP device");
    {
        int dev = 0, lds = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess)
            return nfail(nullptr, CND_EDEVICE, "cnd_net_create: device attributes");
        const size_t need = wg_lds<32, kCP, kCP>();   // the largest of the kernels
        if (need > size_t(lds))
            return nfail(nullptr, CND_EDEVICE, "cnd_net_create: the weight gradients need " + std::to_string(need) +
                                                   " bytes of LDS, the device has " + std::to_string(lds));
    }
    cnd_net *t = new cnd_net;
    t->n = n;
    t->V = n * n * n;
    t->cap = capacity;
    const int64_t V = t->V;
    int r = CND_OK;
    auto ok = [&](int rc) { if (rc) r = rc; return rc == CND_OK; };
    const int64_t S32 = frag_size(C32);
    const int64_t G = wg_slots(n);
    bool good = hipStreamCreateWithFlags(&t->st, hipStreamNonBlocking) == hipSuccess &&
                hipEventCreateWithFlags(&t->done, hipEventDisableTiming) == hipSuccess;
    if (!good) r = nfail(t, CND_EDEVICE, "stream or event creation failed");
    good = good && ok(nalloc(t, &t->p, kNParam)) && ok(nalloc(t, &t->g, kNParam)) && ok(nalloc(t, &t->m1, kNParam)) &&
           ok(nalloc(t, &t->m2, kNParam)) && ok(nalloc(t, &t->gp2, G * kP2)) &&
           ok(nalloc(t, &t->gp1, G * kP1)) && ok(nalloc(t, &t->gp3, G * kP3)) && ok(nalloc(t, &t->b1, G * kCP)) &&
           ok(nalloc(t, &t->b2, G * kCP)) && ok(nalloc(t, &t->b3, G * kCP)) &&
           ok(nalloc(t, &t->slices, kWgSlices * kSlice)) &&
           ok(nalloc(t, &t->W.wf1, frag_size(PAIR))) && ok(nalloc(t, &t->W.wf2, S32)) &&
           ok(nalloc(t, &t->W.wf3, S32)) && ok(nalloc(t, &t->W.wd1, S32)) && ok(nalloc(t, &t->W.wd2, S32)) &&
           ok(nalloc(t, &t->W.wd3, frag_size(SINGLE))) && ok(nalloc(t, &t->x0, V * kC0P)) &&
           ok(nalloc(t, &t->a1, V * kCP)) && ok(nalloc(t, &t->a2, V * kCP)) && ok(nalloc(t, &t->g3, V * kC0P)) &&
           ok(nalloc(t, &t->g2, V * kCP)) && ok(nalloc(t, &t->g1, V * kCP)) && ok(nalloc(t, &t->y, V * kC3)) &&
           ok(nalloc(t, &t->gx, V * kC0)) && ok(nalloc(t, &t->hx, V * kC0)) && ok(nalloc(t, &t->loss, 1)) &&
           ok(nalloc(t, &t->lpart, kConvBlocks)) &&
           ok(nalloc(t, &t->din, int64_t(capacity) * V * kC0P)) && ok(nalloc(t, &t->dtg, int64_t(capacity) * V * kC3));
    if (!good) {
        std::string m = t->err;
        cnd_net_destroy(t);
        return nfail(nullptr, r ? r : CND_ENOMEM, m.empty() ? "allocation failed" : m);
    }
    // He-uniform initial weights, the last layer scaled down so the initial
    // correction is small; zero biases
    std::vector<float> h(kNParam, 0.f);
    std::mt19937_64 rng(seed);
    auto fillu = [&](int off, int cnt, int fan_in, float gain) {
        const float a = gain * std::sqrt(6.0f / float(fan_in));
        std::uniform_real_distribution<float> u(-a, a);
        for (int k = 0; k < cnt; ++k) h[off + k] = u(rng);
    };
    fillu(kOW1, kOB1 - kOW1, kTaps * kC0, 1.0f);
    fillu(kOW2, kOB2 - kOW2, kTaps * kC1, 1.0f);
    fillu(kOW3, kOB3 - kOW3, kTaps * kC2, 0.1f);
    for (int c = 0; c < 5; ++c) { t->nm.in_mean[c] = 0.f; t->nm.in_scale[c] = 1.f; t->nm.out_scale[c] = 1.f; }
    if (hipMemcpy(t->p, h.data(), sizeof(float) * kNParam, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(t->m1, 0, sizeof(float) * kNParam) != hipSuccess ||
        hipMemset(t->m2, 0, sizeof(float) * kNParam) != hipSuccess ||
        hipMemset(t->W.wf1, 0, sizeof(bf16) * frag_size(PAIR)) != hipSuccess ||
        hipMemset(t->W.wf2, 0, sizeof(bf16) * S32) != hipSuccess ||
        hipMemset(t->W.wf3, 0, sizeof(bf16) * S32) != hipSuccess ||
        hipMemset(t->W.wd1, 0, sizeof(bf16) * S32) != hipSuccess ||
        hipMemset(t->W.wd2, 0, sizeof(bf16) * S32) != hipSuccess ||
        hipMemset(t->W.wd3, 0, sizeof(bf16) * frag_size(SINGLE)) != hipSuccess ||
        hipDeviceSynchronize() != hipSuccess || prep(t, t->st) != CND_OK ||
        hipEventRecord(t->done, t->st) != hipSuccess || hipStreamSynchronize(t->st) != hipSuccess) {
        cnd_net_destroy(t);
        return nfail(nullptr, CND_EDEVICE, "initial upload failed");
    }
    *out = t;
    return CND_OK;
}

void cnd_net_destroy(cnd_net *t)
{
    if (!t) return;
    if (t->done) (void)hipEventSynchronize(t->done);
    if (t->st) (void)hipStreamSynchronize(t->st);
    void *ptrs[] = {t->p, t->g, t->m1, t->m2, t->gp2, t->gp1, t->gp3, t->b1, t->b2, t->b3, t->slices, t->W.wf1,
                    t->W.wf2, t->W.wf3, t->W.wd1, t->W.wd2, t->W.wd3, t->x0, t->a1, t->a2, t->g3, t->g2, t->g1, t->y,
                    t->gx, t->hx, t->loss, t->lpart, t->din, t->dtg};
    for (void *p : ptrs) if (p) (void)hipFree(p);
    if (t->done) (void)hipEventDestroy(t->done);
    if (t->st) (void)hipStreamDestroy(t->st);
    delete t;
}

int cnd_net_get_params(cnd_net *t, float *w)
{
    if (!t || !w) return nfail(t, CND_EINVAL, "cnd_net_get_params: bad argument");
    NHIP(t, hipStreamSynchronize(t->st));
    NHIP(t, hipMemcpy(w, t->p, sizeof(float) * kNParam, hipMemcpyDeviceToHost));
    return CND_OK;
}

int cnd_net_set_params(cnd_net *t, const float *w)
{
    if (!t || !w) return nfail(t, CND_EINVAL, "cnd_net_set_params: bad argument");
    NHIP(t, hipEventSynchronize(t->done));
    NHIP(t, hipStreamSynchronize(t->st));
    NHIP(t, hipMemcpy(t->p, w, sizeof(float) * kNParam, hipMemcpyHostToDevice));
    int r;
    if ((r = prep(t, t->st)) || (r = net_end(t, t->st))) return r;
    NHIP(t, hipStreamSynchronize(t->st));
    return CND_OK;
}

int cnd_net_set_norm(cnd_net *t, const double *in_mean, const double *in_scale, const double *out_scale)
{
    if (!t || !in_mean || !in_scale || !out_scale) return nfail(t, CND_EINVAL, "cnd_net_set_norm: bad argument");
    for (int c = 0; c < 5; ++c) {
        if (!(in_scale[c] > 0.0) || !(out_scale[c] > 0.0)) return nfail(t, CND_EINVAL, "cnd_net_set_norm: scales must be > 0");
        t->nm.in_mean[c] = float(in_mean[c]);
        t->nm.in_scale[c] = float(in_scale[c]);
        t->nm.out_scale[c] = float(out_scale[c]);
    }
    return CND_OK;
}

static int coarse_view(cnd_net *t, cnd_ctx *c, int b, CtxView &v, const char *what)
{
    if (ctx_block_view(c, b, v) != CND_OK) return nfail(t, CND_EINVAL, std::string(what) + ": bad context or block");
    if (v.n[0] != t->n + 1 || v.n[1] != t->n + 1 || v.n[2] != t->n + 1)
        return nfail(t, CND_EINVAL, std::string(what) + ": the block must have n+1 points per direction");
    return CND_OK;
}

int cnd_box_filter(cnd_ctx *fine, int bf, cnd_ctx *coarse, int bc)
{
    CtxView F, Cv;
    if (ctx_block_view(fine, bf, F) != CND_OK || ctx_block_view(coarse, bc, Cv) != CND_OK) return CND_EINVAL;
    const int nf = F.n[0] - 1, n = Cv.n[0] - 1;
    if (F.n[1] != F.n[0] || F.n[2] != F.n[0] || Cv.n[1] != Cv.n[0] || Cv.n[2] != Cv.n[0] || n < 1 || nf % n != 0 ||
        (nf / n) % 2 != 0)
        return CND_EINVAL;
    if (hipStreamSynchronize(F.st) != hipSuccess) return CND_EDEVICE;
    const int64_t P = int64_t(n + 1) * (n + 1) * (n + 1);
    hipLaunchKernelGGL(k_box, dim3(blocks_for(P, 256)), dim3(256), 0, Cv.st, F.q, F.NT, F.off, nf, Cv.q, Cv.NT, Cv.off,
                       n, nf / n);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(Cv.st) != hipSuccess) return CND_EDEVICE;
    return CND_OK;
}

int cnd_net_add_pair(cnd_net *t, cnd_ctx *coarse, int bc, cnd_ctx *target, int bt)
{
    if (!t) return nfail(t, CND_EINVAL, "cnd_net_add_pair: null network");
    if (t->npairs >= t->cap) return nfail(t, CND_EINVAL, "cnd_net_add_pair: the pair store is full");
    CtxView C, T;
    int r;
    if ((r = coarse_view(t, coarse, bc, C, "cnd_net_add_pair"))) return r;
    if ((r = coarse_view(t, target, bt, T, "cnd_net_add_pair (target)"))) return r;
    NHIP(t, hipStreamSynchronize(T.st));
    if ((r = net_begin(t, C.st))) return r;
    const int64_t V = t->V;
    hipLaunchKernelGGL(k_pack_state, dim3(blocks_for(V, 256)), dim3(256), 0, C.st, C.q, C.NT, C.off, t->n, t->nm,
                       t->din + int64_t(t->npairs) * V * kC0P);
    hipLaunchKernelGGL(k_target, dim3(blocks_for(V, 256)), dim3(256), 0, C.st, C.q, C.NT, C.off, T.q, T.NT, T.off,
                       t->n, t->nm, t->dtg + int64_t(t->npairs) * V * kC3);
    if ((r = net_end(t, C.st))) return r;
    NHIP(t, hipStreamSynchronize(C.st));
    return t->npairs++;
}

int cnd_net_add_pair_host(cnd_net *t, const float *x, const float *tg)
{
    if (!t || !x || !tg) return nfail(t, CND_EINVAL, "cnd_net_add_pair_host: bad argument");
    if (t->npairs >= t->cap) return nfail(t, CND_EINVAL, "cnd_net_add_pair_host: the pair store is full");
    const int64_t V = t->V;
    hipStream_t st = t->st;
    int r;
    if ((r = net_begin(t, st))) return r;
    NHIP(t, hipMemcpyAsync(t->hx, x, sizeof(float) * V * kC0, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_pack_host_in, dim3(blocks_for(V, 256)), dim3(256), 0, st, t->hx,
                       t->din + int64_t(t->npairs) * V * kC0P, int(V));
    NHIP(t, hipMemcpyAsync(t->dtg + int64_t(t->npairs) * V * kC3, tg, sizeof(float) * V * kC3, hipMemcpyHostToDevice, st));
    if ((r = net_end(t, st))) return r;
    NHIP(t, hipStreamSynchronize(st));
    return t->npairs++;
}

int cnd_net_pairs(const cnd_net *t) { return t ? t->npairs : CND_EINVAL; }

int cnd_net_train(cnd_net *t, int iters, double lr, unsigned long long seed, double *mean_loss)
{
    if (!t || iters < 0 || !(lr > 0.0)) return nfail(t, CND_EINVAL, "cnd_net_train: bad argument");
    if (t->npairs < 1) return nfail(t, CND_ESTATE, "cnd_net_train: no training pairs");
    std::mt19937_64 rng(seed);
    std::uniform_int_distribution<int> pick(0, t->npairs - 1);
    const int64_t V = t->V;
    hipStream_t st = t->st;
    int r;
    if ((r = net_begin(t, st))) return r;
    hipLaunchKernelGGL(k_fill, dim3(1), dim3(256), 0, st, reinterpret_cast<float *>(t->loss), 0.f, 2);
    for (int it = 0; it < iters; ++it) {
        const int k = pick(rng);
        const bf16 *x0 = t->din + int64_t(k) * V * kC0P;
        forward_loss(t, x0, t->dtg + int64_t(k) * V * kC3, t->g3, st);
        const int nl = conv_grid(t->n).blocks;
        if ((r = backward(t, x0, nullptr, st))) return r;
        ++t->adam_t;
        const float c1 = 1.f - std::pow(0.9f, float(t->adam_t)), c2 = 1.f - std::pow(0.999f, float(t->adam_t));
        finish(t, true, float(lr), c1, c2, nl, st);
    }
    double s = 0.0;
    NHIP(t, hipMemcpyAsync(&s, t->loss, sizeof(double), hipMemcpyDeviceToHost, st));
    if ((r = net_end(t, st))) return r;
    NHIP(t, hipStreamSynchronize(st));
    if (mean_loss) *mean_loss = iters > 0 ? s / (double(iters) * 5.0 * double(V)) : 0.0;
    return CND_OK;
}

int cnd_net_eval(cnd_net *t, int first, int count, double *mean_loss)
{
    if (!t || first < 0 || count < 1 || first + count > t->npairs || !mean_loss)
        return nfail(t, CND_EINVAL, "cnd_net_eval: bad range");
    const int64_t V = t->V;
    hipStream_t st = t->st;
    int r;
    if ((r = net_begin(t, st))) return r;
    hipLaunchKernelGGL(k_fill, dim3(1), dim3(256), 0, st, reinterpret_cast<float *>(t->loss), 0.f, 2);
    for (int k = first; k < first + count; ++k) {
        forward_loss(t, t->din + int64_t(k) * V * kC0P, t->dtg + int64_t(k) * V * kC3, nullptr, st);
        hipLaunchKernelGGL(k_loss_add, dim3(1), dim3(256), 0, st, t->lpart, t->loss, conv_grid(t->n).blocks);
    }
    double s = 0.0;
    NHIP(t, hipMemcpyAsync(&s, t->loss, sizeof(double), hipMemcpyDeviceToHost, st));
    if ((r = net_end(t, st))) return r;
    NHIP(t, hipStreamSynchronize(st));
    *mean_loss = s / (double(count) * 5.0 * double(V));
    return CND_OK;
}

int cnd_net_apply(cnd_net *t, cnd_ctx *ctx, int b)
{
    if (!t) return nfail(t, CND_EINVAL, "cnd_net_apply: null network");
    CtxView C;
    int r;
    if ((r = coarse_view(t, ctx, b, C, "cnd_net_apply"))) return r;
    return apply_into(t, C, t->x0, t->a1, t->a2, t->y);
}

int cnd_net_apply_noalloc(cnd_net *t, cnd_ctx *ctx, int b)
{
    if (!t) return nfail(t, CND_EINVAL, "cnd_net_apply_noalloc: null network");
    if (t->n > kScratchN)
        return nfail(t, CND_EINVAL, "cnd_net_apply_noalloc: grid of " + std::to_string(t->n) +
                                        "^3 cells exceeds the scratch limit of " + std::to_string(kScratchN) + "^3");
    CtxView C;
    int r;
    if ((r = coarse_view(t, ctx, b, C, "cnd_net_apply_noalloc"))) return r;
    unsigned char *base = static_cast<unsigned char *>(scratch_address(t));
    if (!base) return CND_EDEVICE;
    // every part is written in full before it is read, so nothing is cleared
    const size_t V = size_t(t->V);
    bf16 *x0 = reinterpret_cast<bf16 *>(base);
    bf16 *a1 = reinterpret_cast<bf16 *>(base + align256(V * 8 * 2));
    bf16 *a2 = reinterpret_cast<bf16 *>(base + align256(V * 8 * 2) + align256(V * 32 * 2));
    float *y = reinterpret_cast<float *>(base + align256(V * 8 * 2) + 2 * align256(V * 32 * 2));
    return apply_into(t, C, x0, a1, a2, y);
}

int cnd_net_forward_host(cnd_net *t, const float *x, float *y)
{
    if (!t || !x || !y) return nfail(t, CND_EINVAL, "cnd_net_forward_host: bad argument");
    const int64_t V = t->V;
    hipStream_t st = t->st;
    int r;
    if ((r = net_begin(t, st))) return r;
    NHIP(t, hipMemcpyAsync(t->hx, x, sizeof(float) * V * kC0, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_pack_host_in, dim3(blocks_for(V, 256)), dim3(256), 0, st, t->hx, t->x0, int(V));
    if ((r = forward(t, t->x0, st))) return r;
    NHIP(t, hipMemcpyAsync(y, t->y, sizeof(float) * V * kC3, hipMemcpyDeviceToHost, st));
    if ((r = net_end(t, st))) return r;
    NHIP(t, hipStreamSynchronize(st));
    return CND_OK;
}

int cnd_net_grad_host(cnd_net *t, const float *x, const float *gy, float *gx, float *gp)
{
    if (!t || !x || !gy || !gx || !gp) return nfail(t, CND_EINVAL, "cnd_net_grad_host: bad argument");
    const int64_t V = t->V;
    hipStream_t st = t->st;
    int r;
    if ((r = net_begin(t, st))) return r;
    NHIP(t, hipMemcpyAsync(t->hx, x, sizeof(float) * V * kC0, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_pack_host_in, dim3(blocks_for(V, 256)), dim3(256), 0, st, t->hx, t->x0, int(V));
    if ((r = forward(t, t->x0, st))) return r;
    NHIP(t, hipMemcpyAsync(t->gx, gy, sizeof(float) * V * kC3, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_pack_host_in, dim3(blocks_for(V, 256)), dim3(256), 0, st, t->gx, t->g3, int(V));
    if ((r = backward(t, t->x0, t->hx, st))) return r;
    finish(t, false, 0.f, 1.f, 1.f, 0, st);
    NHIP(t, hipMemcpyAsync(gx, t->hx, sizeof(float) * V * kC0, hipMemcpyDeviceToHost, st));
    NHIP(t, hipMemcpyAsync(gp, t->g, sizeof(float) * kNParam, hipMemcpyDeviceToHost, st));
    if ((r = net_end(t, st))) return r;
    NHIP(t, hipStreamSynchronize(st));
    return CND_OK;
}

}  // extern "C"
