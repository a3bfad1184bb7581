// unet_kernels.h -- device kernels of the learned coarse-level solver (a 3D
// U-Net on a nodal grid), bfloat16 storage, float32 accumulation.
//
// Activations are channels-last: X[node * C + c], C a multiple of 16, node
// index i fastest.  A 3x3x3 convolution is an implicit GEMM
//     Y[v][n] = sum_{t, c} X[v + d_t][c] * W[n][t * Cin + c]       (K = 27 Cin)
// on the gfx950 matrix cores: v_mfma_f32_16x16x32_bf16 takes a 16 x 32 slice
// of A (16 nodes x 32 of K) and a 32 x 16 slice of B (32 of K x 16 output
// channels), each lane holding 8 consecutive K of one row/column, and
// accumulates a 16 x 16 float32 tile (lane l: rows 4(l/16)..+3, column l%16).
// A K-slice of 8 never straddles two taps because Cin is a multiple of 8.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace aunet {

typedef uint16_t bf16_t;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Threads of the element-wise launches: a constant, as blockDim is read from memory
constexpr int kThreads = 256;
// of those between two levels: a wave each, so that a small level's waves are spread over the CUs
constexpr int kWave = 64;

struct G3 {
    int nx, ny, nz, N;
};

// float -> bfloat16, round to nearest even (finite inputs).
__device__ __forceinline__ bf16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(bf16_t b) { return __uint_as_float(((uint32_t)b) << 16); }

__device__ __forceinline__ void unpack8(const uint4& q, float f[8]) {
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = __uint_as_float(w[i] << 16);
        f[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
    }
}
__device__ __forceinline__ uint4 pack8(const float f[8]) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = (uint32_t)f2bf(f[2 * i]) | ((uint32_t)f2bf(f[2 * i + 1]) << 16);
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// Weights W[n][k] (n a multiple of 16, k < K) are kept in the order in which the
// matrix cores take them: for each 16 of n and 32 of k the 64 lanes' 8 consecutive
// k of one n, so that a wave's load of a step is one run of 1 KB.  The last step is
// filled up with zeros beyond K.
__host__ __device__ inline int frag_steps(int K) { return (K + 31) / 32; }
__host__ __device__ inline size_t frag_index(int K, int n, int k) {
    return ((((size_t)(n >> 4) * frag_steps(K) + (k >> 5)) * 4 + ((k >> 3) & 3)) * 16 + (n & 15)) * 8 + (k & 7);
}
// A weight buffer's elements.
inline size_t frag_size(int K, int n) { return (size_t)(n / 16) * frag_steps(K) * 512; }

// The K rounds of one wave's 16 nodes (from v0 on) x 16*NB output channels (from
// nbase on), starting at k = kfirst and stepping by kstep (a multiple of 32 * KU):
// KU steps of 32 along K per round, the A and B loads of LA rounds issued before
// their MFMAs (a wave waits for memory once per LA rounds; the small levels have
// few waves to hide it), the MFMAs in step order whatever LA is.  CIN > 0 fixes
// the input channels at compile time (0: the argument), so that a step's tap and
// channel need no division.
// The matrix cores want 16 nodes in 16 adjacent lanes.  Loaded so, 4 adjacent
// lanes take 16 bytes each from 4 places, and the gathers bound the kernel.  So 4
// adjacent lanes load one node's 64 bytes of a step, and a move over the LDS
// crossbar brings them to the lanes that multiply them; the weights need no move
// (frag_index).  64 -> 16 channels at 33^3 nodes: 38 us with the matrix cores' own order, 13.2 so.
constexpr int kConvKU = 4;
template <int MT, int NB, int CIN>
__device__ __forceinline__ void conv_rounds(const bf16_t* __restrict__ X, int cin, const bf16_t* __restrict__ Wt,
                                            const G3& g, int v0, int lane, int nbase, int kfirst, int kstep,
                                            f32x4 acc[MT][NB]) {
    constexpr int KU = kConvKU, LA = MT + NB >= 6 ? 1 : 6 / (MT + NB);
    const int Cin = CIN > 0 ? CIN : cin;
    const int K = 27 * Cin;
    const int part = (lane & 3) * 8;  // this lane loads that part of a step of a node
    unsigned taps[MT];                // bit t: the tap is a node of the grid (none: past K or past the last node)
    const bf16_t* xl[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int vox = v0 + 16 * m + (lane >> 2), self = min(vox, g.N - 1);
        const int z = self / (g.nx * g.ny), r = self - z * g.nx * g.ny, y = r / g.nx, x = r - y * g.nx;
        const unsigned mx = (x > 0) | 2u | (x + 1 < g.nx) << 2;
        const unsigned my = (y > 0 ? mx : 0u) | mx << 3 | (y + 1 < g.ny ? mx << 6 : 0u);
        taps[m] = vox < g.N ? (z > 0 ? my : 0u) | my << 9 | (z + 1 < g.nz ? my << 18 : 0u) : 0u;
        xl[m] = X + (size_t)self * Cin + (part & 15);
    }
    const bool hi = part >= 16;
    auto tap_at = [&](int t, int c) {  // channel c of tap t, from xl
        const int dz = t / 9, q = t - 9 * dz, dy = q / 3, dx = q - 3 * dy;
        return (long)(((dz - 1) * g.ny + dy - 1) * g.nx + dx - 1) * Cin + c;
    };
    const bf16_t* wl = Wt + (size_t)(nbase / 16) * frag_steps(K) * 512 + lane * 8;
    const int from = ((lane & 15) * 4 + (lane >> 4)) * 4;  // 4 x the lane that loads what this one multiplies
    auto take = [&](bool ok, const uint4& v) {             // zeros from a lane whose tap is outside
        auto one = [&](uint32_t w) { return (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)(ok ? w : 0u)); };
        return make_uint4(one(v.x), one(v.y), one(v.z), one(v.w));
    };
    for (int k0 = kfirst; k0 < K; k0 += LA * kstep) {
        uint4 a[LA * KU][MT], b[LA * KU][NB];
        unsigned ok[MT] = {};
#pragma unroll
        for (int u = 0; u < LA * KU; ++u) {
            const int ku = k0 + (u / KU) * kstep + 32 * (u % KU);
            if (ku >= K) continue;  // the same for every lane
            // the taps of the step's two halves, the same where Cin is a multiple of 32
            const int t0 = ku / Cin, t1 = CIN > 0 && CIN % 32 == 0 ? t0 : (ku + 16) / Cin;
            const int t = hi ? t1 : t0;
            const long off = hi ? tap_at(t1, ku + 16 - t1 * Cin) : tap_at(t0, ku - t0 * Cin);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const unsigned in = (taps[m] >> t) & 1u;
                ok[m] |= in << u;
                a[u][m] = *reinterpret_cast<const uint4*>(xl[m] + (in ? off : 0L));
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                b[u][nb] = *reinterpret_cast<const uint4*>(wl + ((size_t)nb * frag_steps(K) + (ku >> 5)) * 512);
        }
#pragma unroll
        for (int u = 0; u < LA * KU; ++u) {
            if (k0 + (u / KU) * kstep + 32 * (u % KU) >= K) break;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const bf16x8 A = __builtin_bit_cast(bf16x8, take((ok[m] >> u) & 1u, a[u][m]));
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    acc[m][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, __builtin_bit_cast(bf16x8, b[u][nb]),
                                                                        acc[m][nb], 0, 0, 0);
            }
        }
    }
}

// The biases of a lane's output channels (0 without a bias; the output layer's
// holds yf_ch entries, its Cout is padded to 16).  Loaded before the K rounds: a
// wave that waits for them afterwards waits once more.
template <int NB>
__device__ __forceinline__ void conv_bias(const float* __restrict__ bias, int lane, int nbase, const float* Yf, int yf_ch,
                                          float bv[NB]) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int n = nbase + nb * 16 + (lane & 15);
        bv[nb] = bias && (!Yf || n < yf_ch) ? bias[n] : 0.f;
    }
}
// The epilogue of a 16-node x 16*NB-channel tile: bias, ReLU, and the bf16
// channels-last store, or the float32 component-major one for the output.
template <int NB>
__device__ __forceinline__ void conv_store(const f32x4 acc[NB], const float bv[NB], int Cout, const G3& g, int relu,
                                           int v0, int lane, int nbase, bf16_t* __restrict__ Y, float* __restrict__ Yf,
                                           int yf_ch) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int n = nbase + nb * 16 + (lane & 15);
        if (Yf && n >= yf_ch) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int v = v0 + (lane >> 4) * 4 + e;
            if (v >= g.N) continue;
            float val = acc[nb][e] + bv[nb];
            if (relu) val = fmaxf(val, 0.f);
            if (Yf) {
                Yf[(size_t)n * g.N + v] = val;
            } else {
                Y[(size_t)v * Cout + n] = f2bf(val);
            }
        }
    }
}

// Y = act(conv3(X, W) + bias).  A workgroup is a wave of 16 * MT nodes; blockIdx.y
// selects 16*NB output channels.  Wt is W[n][27 * Cin] in bf16 (frag_index).  bias may be null.
// Yf != null: write float32 component-major Yf[n * N + v] for n < yf_ch
// instead of the bf16 Y (the network output).
template <int MT, int NB, int CIN>
__global__ void __launch_bounds__(64) k_conv_fwd(const bf16_t* __restrict__ X, int Cin, const bf16_t* __restrict__ Wt,
                                                 const float* __restrict__ bias, int Cout, G3 g, int relu,
                                                 bf16_t* __restrict__ Y, float* __restrict__ Yf, int yf_ch) {
    const int lane = threadIdx.x, v0 = blockIdx.x * 16 * MT, nbase = blockIdx.y * 16 * NB;
    float bv[NB];
    conv_bias<NB>(bias, lane, nbase, Yf, yf_ch, bv);
    f32x4 acc[MT][NB];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[m][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    conv_rounds<MT, NB, CIN>(X, Cin, Wt, g, v0, lane, nbase, 0, 32 * kConvKU, acc);
#pragma unroll
    for (int m = 0; m < MT; ++m)
        conv_store<NB>(acc[m], bv, Cout, g, relu, v0 + 16 * m, lane, nbase, Y, Yf, yf_ch);
}

// k_conv_fwd with K split over the KS waves of a workgroup, for the levels
// with few nodes (where k_conv_fwd runs a few dozen waves, each through all
// of K = 27 Cin one round after another).  Every wave of the workgroup takes
// the same 16 nodes and 16*NB channels and every KS-th round of K; wave 0
// adds the others' float32 tiles in wave order through LDS and stores.
template <int NB, int KS, int CIN>
__global__ void __launch_bounds__(64 * KS) k_conv_fwd_ks(const bf16_t* __restrict__ X, int Cin,
                                                         const bf16_t* __restrict__ Wt, const float* __restrict__ bias,
                                                         int Cout, G3 g, int relu, bf16_t* __restrict__ Y,
                                                         float* __restrict__ Yf, int yf_ch) {
    __shared__ f32x4 part[KS - 1][NB][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int v0 = blockIdx.x * 16;
    const int nbase = blockIdx.y * 16 * NB;
    float bv[NB];
    conv_bias<NB>(bias, lane, nbase, Yf, yf_ch, bv);
    f32x4 acc1[1][NB], *acc = acc1[0];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    conv_rounds<1, NB, CIN>(X, Cin, Wt, g, v0, lane, nbase, wave * 32 * kConvKU, 32 * kConvKU * KS, acc1);
    if (wave > 0) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) part[wave - 1][nb][lane] = acc[nb];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < KS - 1; ++w)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[nb] += part[w][nb][lane];
    conv_store<NB>(acc, bv, Cout, g, relu, v0, lane, nbase, Y, Yf, yf_ch);
}

// --- Weight and bias gradients ---------------------------------------------
// dW[co][t][ci] = sum_v dZ[v][co] X[v + d_t][ci] reduces over nodes, which are
// the MFMA K dimension: a lane holds 8 consecutive K of one channel.  The
// activations are channels-last, where those 8 are strided two-byte loads, so
// both operands are first transposed into groups of 8 nodes of a row (the last one
// filled up with zeros): group q = row n8 + i / 8, row = z ny + y, of 16 channels
// in a run of 256 bytes (row_group), so that a wave's load of 4 groups of 16
// channels is 1 KB in a row whichever tap it is for; as T[c][row][i] the 16 lanes
// took 16 bytes from 16 places, which bound the kernel.  X is kept three times,
// shifted by -1, 0 and 1 along i, so that every tap is an aligned 16-byte load.
// At 33^3 nodes, 15 layers: 231 us for the three kernels (wgrad 8.3 us and the
// transposes 5.1 us a layer, finish 30.5 us), where gathers of two bytes a lane, up
// to 1123 partials a weight summed by one thread each, a mask, a bias and an
// unpacking launch took 2112 us.
__host__ __device__ inline size_t row_group(size_t c, long q, long ngroup) {
    return (((c >> 4) * ngroup + q) * 16 + (c & 15)) * 8;
}

// Both transposes of a layer, one thread per (group of 8 nodes, channel); the first
// nbz workgroups take dZ, the others X (4.1 and 4.5 us a layer as two launches,
// 5.1 us as one).
// dZ: the gradient dY of the layer's output masked by its ReLU (Y the output; null:
// no ReLU), in place, its transpose Tz, and the block's sums per channel (the bias
// gradient's partials, bpart[block][C]).  C is a power of two, at most 128.
// X: its three shifted transposes, Tx[s][c][row][i] = X[row][i + s - 1][c] (channel s Cin + c).
__global__ void __launch_bounds__(kThreads) k_wgrad_rows(bf16_t* __restrict__ dY, const bf16_t* __restrict__ Y, int C,
                                                         const bf16_t* __restrict__ X, int Cin, int nx, int n8,
                                                         long ngroup, unsigned nbz, bf16_t* __restrict__ Tz,
                                                         bf16_t* __restrict__ Tx, float* __restrict__ bpart) {
    __shared__ float sh[kThreads];
    if (blockIdx.x >= nbz) {
        const long t = (long)(blockIdx.x - nbz) * kThreads + threadIdx.x;
        const long q = t / Cin;
        if (q >= ngroup) return;
        const int c = (int)(t - q * Cin);
        const long row = q / n8;
        const int i0 = (int)(q - row * n8) * 8;
        uint32_t v[10];
#pragma unroll
        for (int e = 0; e < 10; ++e) {
            const int i = i0 + e - 1;
            const bool in = i >= 0 && i < nx;
            const uint32_t x = X[((size_t)row * nx + (in ? i : 0)) * Cin + c];
            v[e] = in ? x : 0u;
        }
#pragma unroll
        for (int s = 0; s < 3; ++s)
            *reinterpret_cast<uint4*>(Tx + row_group((size_t)s * Cin + c, q, ngroup)) =
                make_uint4(v[s] | (v[s + 1] << 16), v[s + 2] | (v[s + 3] << 16), v[s + 4] | (v[s + 5] << 16),
                           v[s + 6] | (v[s + 7] << 16));
        return;
    }
    const int c = (int)threadIdx.x & (C - 1), sub = (int)threadIdx.x / C, nsub = kThreads / C;
    float sum = 0.f;
    for (long q = (long)blockIdx.x * nsub + sub; q < ngroup; q += (long)nbz * nsub) {
        const long row = q / n8;
        const int i0 = (int)(q - row * n8) * 8;
        const size_t at = ((size_t)row * nx + i0) * C + c;
        uint32_t v[8], y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const size_t o = at + (size_t)(i0 + e < nx ? e : 0) * C;  // in the row
            v[e] = dY[o];
            y[e] = Y ? Y[o] : 1u;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const bool in = i0 + e < nx, pos = (y[e] & 0x7FFFu) != 0 && !(y[e] & 0x8000u);
            v[e] = in && pos ? v[e] : 0u;
            if (Y && in) dY[at + (size_t)e * C] = (bf16_t)v[e];
            sum += bf2f((bf16_t)v[e]);
        }
        *reinterpret_cast<uint4*>(Tz + row_group(c, q, ngroup)) =
            make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
    }
    sh[threadIdx.x] = sum;
    __syncthreads();
    if (sub == 0) {
        for (int w = 1; w < nsub; ++w) sum += sh[w * C + c];
        bpart[(size_t)blockIdx.x * C + c] = sum;
    }
}
// Partial weight gradient of one 16 x 16 tile of (co, ci), all 27 taps, over the
// blockIdx.y-th part of the node groups: part[chunk][co][t][ci].  4 waves share
// the part's steps of 4 groups (one per 16 lanes); their tiles are added in wave
// order through LDS, each wave a quarter of the taps
// (one wave after the other, wave 0 storing all: 12.0 us a layer, 8.3 so).
constexpr int kWgradWaves = 4;
__global__ void __launch_bounds__(64 * kWgradWaves) k_conv_wgrad(const bf16_t* __restrict__ Tx, int Cin,
                                                                 const bf16_t* __restrict__ Tz, int Cout, int ny, int nz,
                                                                 int n8, int steps, float* __restrict__ part) {
    __shared__ f32x4 red[kWgradWaves][27][64];  // 108 KB: a workgroup has a CU to itself
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ncib = Cin / 16, cib = blockIdx.x % ncib, cob = blockIdx.x / ncib, ch = blockIdx.y;
    const int r16 = lane & 15, grp = lane >> 4;
    const int co = cob * 16 + r16, ci = cib * 16 + r16;
    const long ngroup = (long)ny * nz * n8;
    const bf16_t* zc = Tz + row_group(co, 0, ngroup);
    const bf16_t* xc = Tx + row_group(ci, 0, ngroup);
    const size_t sx = (size_t)Cin * ngroup * 8;  // a shift of Tx
    f32x4 acc[27];
#pragma unroll
    for (int t = 0; t < 27; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto keep = [](bool ok, const uint4& v) {  // zeros where the position is outside the grid
        return make_uint4(ok ? v.x : 0u, ok ? v.y : 0u, ok ? v.z : 0u, ok ? v.w : 0u);
    };
    for (int st = wave; st < steps; st += kWgradWaves) {
        const long q = ((long)ch * steps + st) * 4 + grp;
        const bool in = q < ngroup;
        const long qi = in ? q : 0;
        const int row = (int)(qi / n8);
        const int z = row / ny, y = row - z * ny;
        const bf16x8 A = __builtin_bit_cast(bf16x8, keep(in, *reinterpret_cast<const uint4*>(zc + qi * 128)));
        uint4 bq[3][9];
#pragma unroll
        for (int dz = 0; dz < 3; ++dz)
#pragma unroll
            for (int dy = 0; dy < 3; ++dy) {
                const int zz = z + dz - 1, yy = y + dy - 1;
                const bool ok = in && zz >= 0 && zz < nz && yy >= 0 && yy < ny;
                const bf16_t* xr = xc + (qi + (ok ? ((dz - 1) * ny + dy - 1) * n8 : 0)) * 128;
#pragma unroll
                for (int s = 0; s < 3; ++s) bq[dz][3 * dy + s] = keep(ok, *reinterpret_cast<const uint4*>(xr + s * sx));
            }
#pragma unroll
        for (int t = 0; t < 27; ++t)
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, __builtin_bit_cast(bf16x8, bq[t / 9][t % 9]), acc[t], 0,
                                                             0, 0);
    }
#pragma unroll
    for (int t = 0; t < 27; ++t) red[wave][t][lane] = acc[t];
    __syncthreads();
    // acc[t][e] = D[co_local = 4 grp + e][ci_local = r16]
    for (int t = wave; t < 27; t += kWgradWaves) {
        f32x4 sum = red[0][t][lane];
#pragma unroll
        for (int w = 1; w < kWgradWaves; ++w) sum += red[w][t][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            part[(((size_t)ch * Cout + cob * 16 + grp * 4 + e) * 27 + t) * Cin + ci] = sum[e];
    }
}
// Every layer's gradient from its partials, in the canonical parameter order:
// grad[0 .. 27 cin cout) the weights from part[nchunk][coutp][27][cinp], then the
// cout biases from bpart[nb][coutp].  64 entries a workgroup, 4 threads an entry,
// each every 4th partial, added in order.  One launch, layer l from workgroup
// first[l] on (5.3 us a layer as 15 launches, 30.5 us for all).
constexpr int kMaxConv = 15;
struct FinishLayers {
    int n;
    unsigned first[kMaxConv + 1];
    const float *part[kMaxConv], *bpart[kMaxConv];
    float* grad[kMaxConv];
    int nchunk[kMaxConv], cin[kMaxConv], cout[kMaxConv], cinp[kMaxConv], coutp[kMaxConv], nb[kMaxConv];
};
__global__ void __launch_bounds__(kThreads) k_wgrad_finish(FinishLayers F) {
    __shared__ float sh[4][64];
    int l = 0;
    while (blockIdx.x >= F.first[l + 1]) ++l;  // the grid has first[n] workgroups
    const int cin = F.cin[l], cout = F.cout[l], cinp = F.cinp[l], coutp = F.coutp[l], nchunk = F.nchunk[l], nb = F.nb[l];
    const long nw = 27L * cin * cout, e = (long)(blockIdx.x - F.first[l]) * 64 + (threadIdx.x & 63);
    const int sl = threadIdx.x >> 6;
    float s = 0.f;
    if (e < nw) {
        const long q = e / cin;
        const float* p = F.part[l] + q * cinp + (e - q * cin);  // q = co 27 + t
        const long M = 27L * cinp * coutp;
#pragma unroll 4
        for (int c = sl; c < nchunk; c += 4) s += p[c * M];
    } else if (e < nw + cout) {
        const float* p = F.bpart[l] + (e - nw);
#pragma unroll 4
        for (int c = sl; c < nb; c += 4) s += p[(size_t)c * coutp];
    }
    sh[sl][threadIdx.x & 63] = s;
    __syncthreads();
    if (sl == 0 && e < nw + cout) F.grad[l][e] = ((s + sh[1][threadIdx.x]) + sh[2][threadIdx.x]) + sh[3][threadIdx.x];
}

// Canonical float32 W[Cout][27][Cin] -> bf16 Wt[Coutp][27 * Cinp] (zero
// padded) and the flipped transpose Wb[Cinp][27 * Coutp],
// Wb[ci][t][co] = W[co][26 - t][ci], used by the input gradient, both in the order
// of frag_index.  Every layer in one launch: layer l takes the threads from first[l] on.
struct PackLayers {
    int n;
    long first[kMaxConv + 1];
    const float* W[kMaxConv];
    int cin[kMaxConv], cout[kMaxConv], cinp[kMaxConv], coutp[kMaxConv];
    bf16_t *wt[kMaxConv], *wb[kMaxConv];
};
__global__ void __launch_bounds__(kThreads) k_pack_weights(PackLayers P) {
    const long e = (long)blockIdx.x * kThreads + threadIdx.x;
    if (e >= P.first[P.n]) return;
    int l = 0;
    while (e >= P.first[l + 1]) ++l;
    const unsigned i = (unsigned)(e - P.first[l]), cinp = P.cinp[l];
    const unsigned q = i / cinp, ci = i - q * cinp, co = q / 27, t = q - co * 27;
    const float w = ((int)ci < P.cin[l] && (int)co < P.cout[l]) ? P.W[l][((size_t)co * 27 + t) * P.cin[l] + ci] : 0.f;
    const bf16_t b = f2bf(w);
    P.wt[l][frag_index(27 * (int)cinp, (int)co, (int)(t * cinp + ci))] = b;
    P.wb[l][frag_index(27 * P.coutp[l], (int)ci, (int)((26 - t) * P.coutp[l] + co))] = b;
}

// Full weighting with scale: Y[I][c] = scale * sum_d w(d) X[2I + d][c],
// w(d) = prod_a (1 - |d_a| / 2), zero outside the fine grid.  X has ld channels a
// node, the first C of them are taken.  2 channels per thread: the grids are small
// and a wave's own instructions the longest part (33^3 to 17^3, 16 channels: 5.8 us with 8
// channels a thread, 3.2 with 2).  All 27 loads leave
// before the sums (in tap order; a position outside the grid reads the node itself
// and adds 0).
__global__ void __launch_bounds__(kWave) k_down(const bf16_t* __restrict__ X, int ld, int C, G3 gf, G3 gc, float scale,
                                                bf16_t* __restrict__ Y) {
    const unsigned c2 = C / 2;
    const unsigned i = blockIdx.x * kWave + threadIdx.x;
    if (i >= (unsigned)gc.N * c2) return;
    const unsigned I = i / c2, q = i - I * c2, nxy = (unsigned)gc.nx * gc.ny;
    const int z = 2 * (int)(I / nxy), r = I % nxy, y = 2 * (r / gc.nx), x = 2 * (r % gc.nx);
    const unsigned mx = (x > 0) | 2u | (x + 1 < gf.nx) << 2;
    const unsigned my = (y > 0 ? mx : 0u) | mx << 3 | (y + 1 < gf.ny ? mx << 6 : 0u);
    const unsigned in = (z > 0 ? my : 0u) | my << 9 | (z + 1 < gf.nz ? my << 18 : 0u);  // bit t: the tap is in the grid
    const bf16_t* xl = X + ((size_t)(z * gf.ny + y) * gf.nx + x) * ld + 2 * q;
    uint32_t v[27];
#pragma unroll
    for (int t = 0; t < 27; ++t) {
        const long off = (long)(((t / 9 - 1) * gf.ny + t / 3 % 3 - 1) * gf.nx + t % 3 - 1) * ld;
        v[t] = *reinterpret_cast<const uint32_t*>(xl + ((in >> t) & 1u ? off : 0L));
    }
    float lo = 0.f, hi = 0.f;
#pragma unroll
    for (int t = 0; t < 27; ++t) {
        const float w = (t % 3 != 1 ? 0.5f : 1.f) * (t / 3 % 3 != 1 ? 0.5f : 1.f) * (t / 9 != 1 ? 0.5f : 1.f);
        const uint32_t u = (in >> t) & 1u ? v[t] : 0u;
        lo += w * __uint_as_float(u << 16);
        hi += w * __uint_as_float(u & 0xFFFF0000u);
    }
    *reinterpret_cast<uint32_t*>(Y + (size_t)I * C + 2 * q) =
        (uint32_t)f2bf(lo * scale) | ((uint32_t)f2bf(hi * scale) << 16);
}

// The trilinear value of 8 channels at fine node v (x, y, z): w times the sum of
// the 1 to 8 coarse nodes around it, in (z, y, x) order.  All 8 are loaded (those
// of an even coordinate twice) and the repeats left out of the sum.
__device__ __forceinline__ void up_value(const bf16_t* __restrict__ X, int C, const G3& gc, const G3& gf, int v, int q,
                                         float acc[8]) {
    const int z = v / (gf.nx * gf.ny), r = v - z * gf.nx * gf.ny, y = r / gf.nx, x = r - y * gf.nx;
    uint4 u[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int xs = (x + (e & 1)) >> 1, ys = (y + ((e >> 1) & 1)) >> 1, zs = (z + (e >> 2)) >> 1;
        u[e] = *reinterpret_cast<const uint4*>(X + ((size_t)(zs * gc.ny + ys) * gc.nx + xs) * C + 8 * q);
    }
    const int n = ((x & 1) + 1) * ((y & 1) + 1) * ((z & 1) + 1);
    const float w = 1.f / (float)n;
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const bool use = (!(e & 1) || (x & 1)) && (!(e & 2) || (y & 1)) && (!(e & 4) || (z & 1));
        float f[8];
        unpack8(u[e], f);
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] = use ? acc[k] + w * f[k] : acc[k];
    }
}
// Interpolation with scale and addend: Y[i][c] = scale * (P X)[i][c] + add[i][c],
// add with ld channels a node, its C from channel off on.
__global__ void __launch_bounds__(kWave) k_up_add(const bf16_t* __restrict__ X, int C, G3 gc, G3 gf, float scale,
                                                     const bf16_t* __restrict__ add, int ld, int off,
                                                     bf16_t* __restrict__ Y) {
    const unsigned c8 = C / 8;
    const unsigned i = blockIdx.x * kWave + threadIdx.x;
    if (i >= (unsigned)gf.N * c8) return;
    const int v = (int)(i / c8), q = (int)(i - v * c8);
    float ad[8], acc[8];
    const uint4 a = *reinterpret_cast<const uint4*>(add + (size_t)v * ld + off + 8 * q);
    up_value(X, C, gc, gf, v, q, acc);
    unpack8(a, ad);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = scale * acc[e] + ad[e];
    *reinterpret_cast<uint4*>(Y + (size_t)v * C + 8 * q) = pack8(acc);
}
// The decoder's input Y[v] = [(P X)[v] (C channels), E[v] (Ce channels)].
__global__ void __launch_bounds__(kWave) k_up_concat(const bf16_t* __restrict__ X, int C, G3 gc, G3 gf,
                                                        const bf16_t* __restrict__ E, int Ce, bf16_t* __restrict__ Y) {
    const unsigned c8 = (C + Ce) / 8;
    const unsigned i = blockIdx.x * kWave + threadIdx.x;
    if (i >= (unsigned)gf.N * c8) return;
    const int v = (int)(i / c8), q = (int)(i - v * c8);
    uint4 val;
    if (8 * q < C) {
        float acc[8];
        up_value(X, C, gc, gf, v, q, acc);
        val = pack8(acc);
    } else {
        val = *reinterpret_cast<const uint4*>(E + (size_t)v * Ce + 8 * q - C);
    }
    *reinterpret_cast<uint4*>(Y + (size_t)v * (C + Ce) + 8 * q) = val;
}

// Component-major float32 in[c * N + v] (c < n) -> bf16 X[v * Cp + c] (zero
// padded), 64 nodes x 16 channels a workgroup (blockIdx.y: the channels) through
// LDS: nodes fastest on the way in, channels on the way out.
__global__ void __launch_bounds__(kThreads) k_pack_soa(const float* __restrict__ in, int n, int Cp, int N,
                                                       bf16_t* __restrict__ X) {
    __shared__ bf16_t sh[64][16 + 2];
    const int v0 = blockIdx.x * 64, c0 = blockIdx.y * 16, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int c = c0 + 4 * k + w, v = v0 + lane;
        sh[lane][4 * k + w] = c < n && v < N ? f2bf(in[(size_t)c * N + v]) : (bf16_t)0;
    }
    __syncthreads();
    const int v = threadIdx.x >> 2, q = (threadIdx.x & 3) * 4;
    if (v0 + v >= N) return;
    const bf16_t* p = &sh[v][q];
    *reinterpret_cast<uint2*>(X + (size_t)(v0 + v) * Cp + c0 + q) =
        make_uint2(p[0] | ((uint32_t)p[1] << 16), p[2] | ((uint32_t)p[3] << 16));
}
// bf16 X[v * Cp + c] -> float32 out[c * N + v] for c < n.
__global__ void __launch_bounds__(256) k_unpack_soa(const bf16_t* __restrict__ X, int n, int Cp, int N,
                                                    float* __restrict__ out) {
    const long i = (long)blockIdx.x * kThreads + threadIdx.x;
    if (i >= (long)N * n) return;
    const int v = (int)(i % N), c = (int)(i / N);
    out[i] = bf2f(X[(size_t)v * Cp + c]);
}

// Mean squared error over n components: loss partials and d = 2 (y - t) / (n N).
__global__ void __launch_bounds__(256) k_mse(const float* __restrict__ y, const float* __restrict__ t, long M,
                                             float inv, float* __restrict__ d, float* __restrict__ part) {
    __shared__ float sh[256];
    float s = 0.f;
    for (long i = (long)blockIdx.x * kThreads + threadIdx.x; i < M; i += (long)gridDim.x * kThreads) {
        const float e = y[i] - t[i];
        s += e * e;
        if (d) d[i] = 2.f * e * inv;
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// Adam on float32 parameters (bias-corrected, no weight decay).
__global__ void __launch_bounds__(256) k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                                              float* __restrict__ v, long n, float lr, float b1, float b2, float eps,
                                              float c1, float c2) {
    const long i = (long)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

}  // namespace aunet
