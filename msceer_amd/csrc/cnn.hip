// Near-separatrix classifier: a small 3-D CNN with hand-written kernels.
//
// Input: the value field normalised over the 9x9x9 window centred on each
// vertex (window clamped to the domain): n = (f - mean) / (std + 1e-6).
// Layers (3x3x3 taps, zero padding, channels-last activations in BF16):
//   conv1  1 -> 16, ReLU        (VALU, FP32)
//   conv2 16 -> 32, ReLU        (MFMA 32x32x16 bf16, FP32 accumulation)
//   conv3 32 -> 16, ReLU        (MFMA 16x16x32 bf16, FP32 accumulation)
//   head  16 -> 1, sigmoid      (fused into conv3 for inference)
// Weights are kept in FP32 (Adam state) and packed to BF16 for the
// convolutions; biases and the head stay FP32.  Tap t = (dx+1) + 3(dy+1) +
// 9(dz+1) reads the input at (x+dx, y+dy, z+dz).
//
// Training: weighted binary cross-entropy (mean over voxels), backward by
// transposed convolutions on the same MFMA kernels (taps mirrored, weights
// transposed), weight gradients on VALU with per-block partial sums reduced
// in a fixed order (deterministic), Adam.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "cnn.hpp"
#include "ctx.hpp"

namespace msceer {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kT = 256;

__device__ __forceinline__ uint16_t f2bf(float x) {
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7F800000u) == 0x7F800000u) return (uint16_t)(u >> 16);  // inf / nan
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

struct Geo {
    int X, Y, Z;
    int64_t sxy;
    __host__ __device__ __forceinline__ int64_t verts() const { return sxy * Z; }
};

__device__ __forceinline__ int tap_dx(int t) { return t % 3 - 1; }
__device__ __forceinline__ int tap_dy(int t) { return (t / 3) % 3 - 1; }
__device__ __forceinline__ int tap_dz(int t) { return t / 9 - 1; }

// Tile of a work-group: tiles along x, then y, then z; work-groups are dealt to
// the eight XCDs round robin, so each takes a contiguous run of the tiles and
// neighbours share their halos in one L2.  A launch takes at most kMaxTiles of
// them (a grid holds fewer than 2^32 threads), from `first` on.
struct Tiles {
    uint32_t first, n, x, y;  // of this launch; along x and y
};
struct Tile {
    int x, y, z;
};
constexpr uint32_t kMaxTiles = 1u << 22;
__device__ __forceinline__ Tile tile_of(const Tiles& a) {
    const uint32_t per = a.n / 8u, rem = a.n % 8u, xcd = blockIdx.x % 8u, k = blockIdx.x / 8u;
    const uint32_t t = a.first + (xcd < rem ? xcd * (per + 1u) + k : rem * (per + 1u) + (xcd - rem) * per + k);
    const uint32_t q = t / a.x;
    return Tile{(int)(t % a.x), (int)(q % a.y), (int)(q / a.y)};
}

// ---- local normalisation (separable 9-wide box sums in FP64) ----------------

// Sums along x, then along y, for a tile of 64x16 vertices of one layer: values
// and x sums in LDS.  Absent vertices add zeros, in the order of the window, so
// the sums are those of the present ones alone.  Bound by LDS reads (9 values
// and 3 pairs of doubles per vertex) and the 16 B/vertex written: 41 us at
// 256x192x128; as two passes over memory, with each pair of sums read 9 times
// and coordinates by 64-bit division, 182.
constexpr int kNormX = 64, kNormY = 16;
__global__ void __launch_bounds__(kT) norm_xy_kernel(const float* __restrict__ f, Geo g, Tiles tiles,
                                                     double2* __restrict__ out) {
    __shared__ float sv[kNormY + 8][kNormX + 8];
    __shared__ double2 sx[kNormY + 8][kNormX];
    const Tile t = tile_of(tiles);
    const int x0 = t.x * kNormX, y0 = t.y * kNormY;
    const float* const layer = f + (int64_t)t.z * g.sxy;
    for (int i = threadIdx.x; i < (kNormY + 8) * (kNormX + 8); i += kT) {
        const int ly = i / (kNormX + 8), lx = i % (kNormX + 8), x = x0 + lx - 4, y = y0 + ly - 4;
        const bool in = x >= 0 && x < g.X && y >= 0 && y < g.Y;
        sv[ly][lx] = in ? layer[(int64_t)y * g.X + x] : 0.f;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < (kNormY + 8) * kNormX; i += kT) {
        const int ly = i / kNormX, lx = i % kNormX;
        double s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int d = 0; d < 9; d++) {
            const double a = (double)sv[ly][lx + d];
            s1 += a;
            s2 += a * a;
        }
        sx[ly][lx] = make_double2(s1, s2);
    }
    __syncthreads();
    constexpr int kRows = kNormY * kNormX / kT;  // rows per thread
    const int lx = threadIdx.x % kNormX, ly = threadIdx.x / kNormX * kRows, x = x0 + lx;
    double2 col[kRows + 8];
#pragma unroll
    for (int d = 0; d < kRows + 8; d++) col[d] = sx[ly + d][lx];
    if (x >= g.X) return;
#pragma unroll
    for (int j = 0; j < kRows; j++) {
        const int y = y0 + ly + j;
        if (y >= g.Y) break;
        double s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int d = 0; d < 9; d++) {
            s1 += col[j + d].x;
            s2 += col[j + d].y;
        }
        out[(int64_t)t.z * g.sxy + (int64_t)y * g.X + x] = make_double2(s1, s2);
    }
}

__device__ __forceinline__ int win_count(int c, int n) {
    const int lo = c - 4 < 0 ? 0 : c - 4, hi = c + 4 >= n ? n - 1 : c + 4;
    return hi - lo + 1;
}

// Sums along z and the normalised value, kNormZ vertices up per thread: 16 sums
// read for 8 vertices.  Bound by the FP64 division and square root: 43 us at
// 256x192x128 (63 with 9 reads a vertex).
constexpr int kNormZ = 8;
__global__ void __launch_bounds__(kT)
norm_z_kernel(const double2* __restrict__ in, const float* __restrict__ f, Geo g, Tiles tiles, float* __restrict__ out) {
    const Tile t = tile_of(tiles);
    const int x = t.x * 64 + (int)(threadIdx.x & 63u), y = t.y * (kT / 64) + (int)(threadIdx.x >> 6), z0 = t.z * kNormZ;
    if (x >= g.X || y >= g.Y) return;
    const int64_t v0 = (int64_t)z0 * g.sxy + (int64_t)y * g.X + x;
    double2 col[kNormZ + 8];
#pragma unroll
    for (int d = 0; d < kNormZ + 8; d++) {
        const int z = z0 + d - 4;
        col[d] = z >= 0 && z < g.Z ? in[v0 + (int64_t)(d - 4) * g.sxy] : make_double2(0.0, 0.0);
    }
    const double cxy = (double)win_count(x, g.X) * win_count(y, g.Y);
#pragma unroll
    for (int j = 0; j < kNormZ; j++) {
        const int z = z0 + j;
        if (z >= g.Z) break;
        double s1 = 0.0, s2 = 0.0;
#pragma unroll
        for (int d = 0; d < 9; d++) {
            s1 += col[j + d].x;
            s2 += col[j + d].y;
        }
        const int64_t v = v0 + (int64_t)j * g.sxy;
        const double cnt = cxy * win_count(z, g.Z);
        const double mean = s1 / cnt;
        double var = s2 / cnt - mean * mean;
        if (var < 0.0) var = 0.0;
        out[v] = (float)(((double)f[v] - mean) / (sqrt(var) + 1e-6));
    }
}

// Two values to BF16, nearest even (no NaN reaches it).
__device__ __forceinline__ uint32_t pack_bf(float lo, float hi) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)lo) |
           (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)hi) << 16;
}
__device__ __forceinline__ float relu(float v) { return v > 0.f ? v : 0.f; }  // (of NaN: 0)

// ---- conv1: 1 -> 16, ReLU (VALU) --------------------------------------------

// A wave takes 64 vertices along x by 4 rows: each tap's 16 weights, read from
// LDS by all lanes at once, serve the four.  Bound by VALU issue, 432 FMAs a
// vertex: 95 us at 256x192x128.  With one vertex per lane and each weight read
// for it alone it was bound by the LDS reads, 466; with the weights of two rows
// by scalar loads, which the compiler moves to the front and spills, 169.
constexpr int kC1Rows = 4;
__global__ void __launch_bounds__(kT)
conv1_kernel(const float* __restrict__ xin, Geo g, Tiles tiles, const float* __restrict__ w1 /*[27][16] bf16-rounded*/,
             const float* __restrict__ b1, uint16_t* __restrict__ a1) {
    __shared__ __attribute__((aligned(16))) float sw[27 * 16];
    for (int i = threadIdx.x; i < 27 * 16; i += kT) sw[i] = w1[i];
    __syncthreads();
    const Tile t = tile_of(tiles);
    const int x = t.x * 64 + (int)(threadIdx.x & 63u), y0 = t.y * kC1Rows;
    const int z = t.z * (kT / 64) + (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (z >= g.Z) return;
    const int xc = min(x, g.X - 1), xl = max(xc - 1, 0), xr = min(xc + 1, g.X - 1);
    const bool okl = x > 0, okr = x + 1 < g.X;
    float acc[kC1Rows][16];
#pragma unroll
    for (int c = 0; c < 16; c++)
#pragma unroll
        for (int j = 0; j < kC1Rows; j++) acc[j][c] = b1[c];
#pragma unroll 1
    for (int dz = 0; dz < 3; dz++) {
        const int zz = z + dz - 1;
        const bool zok = zz >= 0 && zz < g.Z;
        const float* const layer = xin + (int64_t)(zok ? zz : z) * g.sxy;
        float nv[kC1Rows + 2][3];
#pragma unroll
        for (int i = 0; i < kC1Rows + 2; i++) {
            const int yy = y0 + i - 1;
            const bool yok = yy >= 0 && yy < g.Y, ok = zok && yok;  // the same in every lane
            const float* const row = layer + (int64_t)(yok ? yy : y0) * g.X;
            const float l = row[xl], c = row[xc], r = row[xr];
            nv[i][0] = ok && okl ? l : 0.f;
            nv[i][1] = ok ? c : 0.f;
            nv[i][2] = ok && okr ? r : 0.f;
        }
#pragma unroll
        for (int k = 0; k < 9; k++) {
            const float4* const wk = reinterpret_cast<const float4*>(sw + (dz * 9 + k) * 16);
            const float4 w0 = wk[0], w4 = wk[1], w8 = wk[2], wc = wk[3];
            const float w[16] = {w0.x, w0.y, w0.z, w0.w, w4.x, w4.y, w4.z, w4.w,
                                 w8.x, w8.y, w8.z, w8.w, wc.x, wc.y, wc.z, wc.w};
#pragma unroll
            for (int c = 0; c < 16; c++)
#pragma unroll
                for (int j = 0; j < kC1Rows; j++) acc[j][c] = fmaf(w[c], nv[j + k / 3][k % 3], acc[j][c]);
        }
    }
    if (x >= g.X) return;
#pragma unroll
    for (int j = 0; j < kC1Rows; j++) {
        if (y0 + j >= g.Y) break;
        uint32_t p[8];
#pragma unroll
        for (int c = 0; c < 8; c++) p[c] = pack_bf(relu(acc[j][2 * c]), relu(acc[j][2 * c + 1]));
        uint4* o = reinterpret_cast<uint4*>(a1 + ((int64_t)z * g.sxy + (int64_t)(y0 + j) * g.X + x) * 16);
        o[0] = make_uint4(p[0], p[1], p[2], p[3]);
        o[1] = make_uint4(p[4], p[5], p[6], p[7]);
    }
}

// ---- MFMA convolutions ------------------------------------------------------

enum ConvMode : int {
    kFwd = 0,      // out = relu(acc + bias), BF16
    kBwd = 1,      // out = acc * (gate > 0), BF16 (transposed convolution of a gradient)
    kFwdHead = 2,  // prob = sigmoid(head . relu(acc + bias)), FP32 (conv3 only)
};

__device__ __forceinline__ bf16x8 load8(const uint16_t* p) {
    const uint4 u = *reinterpret_cast<const uint4*>(p);
    return __builtin_bit_cast(bf16x8, u);
}

// Two values of a gradient to BF16 where the activations are positive.
__device__ __forceinline__ uint32_t gated(uint32_t gate, float lo, float hi) {
    return (bf2f((uint16_t)gate) > 0.f ? (uint32_t)f2bf(lo) : 0u) |
           (bf2f((uint16_t)(gate >> 16)) > 0.f ? (uint32_t)f2bf(hi) : 0u) << 16;
}

// Both convolutions: a work-group computes 32x16 vertices of `layers` layers,
// each wave several rows along y of one x tile.  It runs up the input layers:
// 34x18 vertices of one are staged in LDS (the next one's loads are in flight
// meanwhile) and serve the three output layers they are taps of, two of which
// a wave keeps between steps.  Per layer of taps a wave holds its 9 weight
// operands and runs over the input rows; an input row (three LDS reads, one per
// dx) serves the up to three output rows it is a tap of.  So every output still
// sums its taps in order.  The weights are the A operand and the vertices the
// columns: a lane then holds several channels of one vertex, and stores (or
// sums, for the head) them together.  Bound by LDS reads and MFMA, about even,
// with the memory traffic behind them (256x192x128: 0.6 GB for 16 -> 32, 0.4 GB
// for 32 -> 16): 164 and 178 us, of which the MFMAs alone take 69 each.  Without
// the run along z, three layers staged per output layer: 248 and 265; without
// LDS, bound by the cache's accesses: 345 and 345; a wave per row with a load per
// tap and MFMA, vertices as rows and 2-byte stores: 553 and 835.
constexpr int kCx = 32, kCy = 16;

// One layer of a tile with its rim for the work-group: kC channels, zero where
// there is no vertex.
template <int kC>
struct Stage {
    static constexpr int kPer = kC / 8, kAll = (kCx + 2) * (kCy + 2) * kPer, kK = (kAll + kT - 1) / kT;
    int32_t at[kK];  // 16-byte pieces from the layer's tile origin, -1: none
    uint4 u[kK];
    __device__ Stage(const Geo& g, int x0, int y0) {
#pragma unroll
        for (int k = 0; k < kK; k++) {
            const int i = (int)threadIdx.x + k * kT, v = i / kPer, x = x0 + v % (kCx + 2) - 1, y = y0 + v / (kCx + 2) - 1;
            const bool in = i < kAll && x >= 0 && x < g.X && y >= 0 && y < g.Y;
            at[k] = in ? ((y - max(y0 - 1, 0)) * g.X + x) * kPer + i % kPer : -1;  // (< 18 * 2^16 * 4)
        }
    }
    // tile: the layer's row max(y0 - 1, 0); ok: the layer is there
    __device__ __forceinline__ void load(const uint4* __restrict__ tile, bool ok) {
#pragma unroll
        for (int k = 0; k < kK; k++) {
            u[k] = make_uint4(0u, 0u, 0u, 0u);
            if (ok && at[k] >= 0) u[k] = tile[at[k]];
        }
    }
    __device__ __forceinline__ void store(uint4* lds) const {
#pragma unroll
        for (int k = 0; k < kK; k++) {
            const int i = (int)threadIdx.x + k * kT;
            if (i < kAll) lds[i] = u[k];
        }
    }
};

// conv 16 -> 32, a wave 32 vertices x kC2Rows rows, MFMA 32x32x16 (wave64):
// A[row = lane%32][k = 8*(lane/32) .. +8], B[k = 8*(lane/32) .. +8][col = lane%32],
// D[i]: row 8*(i/4) + 4*(lane/32) + i%4, col lane%32.  Row m of A is output
// channel 16*((m/4)%2) + 4*(m/8) + m%4, so D[i] is channel 16*(lane/32) + i.
constexpr int kC2Rows = 4;  // of 16 for four waves
template <int kMode>
__global__ void __launch_bounds__(kT)
conv16to32_kernel(const uint16_t* __restrict__ in, Geo g, Tiles tiles, int layers, const uint16_t* __restrict__ w /*[27][32][16]*/,
                  const float* __restrict__ bias, const uint16_t* __restrict__ gate, uint16_t* __restrict__ out) {
    __shared__ __attribute__((aligned(16))) uint16_t sw[27 * 32 * 16];
    __shared__ __attribute__((aligned(16))) uint16_t sv[(kCx + 2) * (kCy + 2) * 16];
    __shared__ float sb[32];
    if (kMode == kFwd && threadIdx.x < 32) sb[threadIdx.x] = bias[threadIdx.x];
    for (int i = threadIdx.x; i < 27 * 32 * 16 / 8; i += kT)
        reinterpret_cast<uint4*>(sw)[i] = reinterpret_cast<const uint4*>(w)[i];
    const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
    const int wave = (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Tile t = tile_of(tiles);
    const int x = t.x * kCx + r, y0 = t.y * kCy + wave * kC2Rows;
    const int z0 = t.z * layers, z1 = min(z0 + layers, g.Z);
    const uint16_t* const wl = sw + (16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3)) * 16 + 8 * h;
    const uint16_t* const vl = sv + (wave * kC2Rows * (kCx + 2) + r) * 16 + 8 * h;
    Stage<16> stage(g, t.x * kCx, t.y * kCy);
    const uint4* const tile = reinterpret_cast<const uint4*>(in + (int64_t)max(t.y * kCy - 1, 0) * g.X * 16);
    auto load = [&](int z) { stage.load(tile + (int64_t)z * g.sxy * 2, z >= 0 && z < g.Z); };
    // adds the taps of layer dz that lie in the staged input layer
    auto taps = [&](f32x16 acc[kC2Rows], int dz) {
        bf16x8 wt[9];
#pragma unroll
        for (int k = 0; k < 9; k++) wt[k] = load8(wl + (dz * 9 + k) * 512);
#pragma unroll
        for (int i = 0; i < kC2Rows + 2; i++)
#pragma unroll
            for (int dx = 0; dx < 3; dx++) {
                const bf16x8 v = load8(vl + (i * (kCx + 2) + dx) * 16);
#pragma unroll
                for (int dy = 0; dy < 3; dy++)
                    if (i - dy >= 0 && i - dy < kC2Rows)
                        acc[i - dy] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wt[3 * dy + dx], v, acc[i - dy], 0, 0, 0);
            }
    };
    auto emit = [&](const f32x16 acc[kC2Rows], int z) {
        if (x >= g.X) return;
#pragma unroll
        for (int j = 0; j < kC2Rows; j++) {
            if (y0 + j >= g.Y) break;
            const int64_t at = ((int64_t)z * g.sxy + (int64_t)(y0 + j) * g.X + x) * 32 + 16 * h;
            uint32_t p[8];
            if (kMode == kFwd) {
                const float* const b = sb + 16 * h;
#pragma unroll
                for (int i = 0; i < 8; i++)
                    p[i] = pack_bf(relu(acc[j][2 * i] + b[2 * i]), relu(acc[j][2 * i + 1] + b[2 * i + 1]));
            } else {
                const uint4 g0 = reinterpret_cast<const uint4*>(gate + at)[0], g1 = reinterpret_cast<const uint4*>(gate + at)[1];
                const uint32_t gs[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
                for (int i = 0; i < 8; i++) p[i] = gated(gs[i], acc[j][2 * i], acc[j][2 * i + 1]);
            }
            uint4* const o = reinterpret_cast<uint4*>(out + at);
            o[0] = make_uint4(p[0], p[1], p[2], p[3]);
            o[1] = make_uint4(p[4], p[5], p[6], p[7]);
        }
    };
    f32x16 a[kC2Rows] = {}, b[kC2Rows] = {};  // of the layers below and at the input layer
    load(z0 - 1);
#pragma unroll 1
    for (int z = z0 - 1; z <= z1; z++) {
        __syncthreads();
        stage.store(reinterpret_cast<uint4*>(sv));
        if (z < z1) load(z + 1);
        __syncthreads();
        if (z > z0) {
            taps(a, 2);
            emit(a, z - 1);
        }
        if (z >= z0 && z < z1) {
#pragma unroll
            for (int j = 0; j < kC2Rows; j++) a[j] = b[j];
            taps(a, 1);
        }
        if (z + 1 < z1) {
#pragma unroll
            for (int j = 0; j < kC2Rows; j++) b[j] = f32x16{};
            taps(b, 0);
        }
    }
}

// conv 32 -> 16, a wave 16 vertices x kC3Rows rows, MFMA 16x16x32:
// A[row = lane%16][k = 8*(lane/16) .. +8], B[k = 8*(lane/16) .. +8][col = lane%16],
// D[i]: row (channel) 4*(lane/16) + i, col (vertex) lane%16.
constexpr int kC3Rows = 8;  // four waves: 2 x 2
template <int kMode>
__global__ void __launch_bounds__(kT)
conv32to16_kernel(const uint16_t* __restrict__ in, Geo g, Tiles tiles, int layers, const uint16_t* __restrict__ w /*[27][16][32]*/,
                  const float* __restrict__ bias, const float* __restrict__ head /*[16] + bias*/,
                  const uint16_t* __restrict__ gate, uint16_t* __restrict__ out, float* __restrict__ prob) {
    __shared__ __attribute__((aligned(16))) uint16_t sw[27 * 16 * 32];
    __shared__ __attribute__((aligned(16))) uint16_t sv[(kCx + 2) * (kCy + 2) * 32];
    for (int i = threadIdx.x; i < 27 * 16 * 32 / 8; i += kT)
        reinterpret_cast<uint4*>(sw)[i] = reinterpret_cast<const uint4*>(w)[i];
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int wave = (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Tile t = tile_of(tiles);
    const int lx = (wave & 1) * 16, ly = (wave >> 1) * kC3Rows;
    const int x = t.x * kCx + lx + r, y0 = t.y * kCy + ly;
    const int z0 = t.z * layers, z1 = min(z0 + layers, g.Z);
    const uint16_t* const wl = sw + r * 32 + 8 * q;
    const uint16_t* const vl = sv + (ly * (kCx + 2) + lx + r) * 32 + 8 * q;
    Stage<32> stage(g, t.x * kCx, t.y * kCy);
    const uint4* const tile = reinterpret_cast<const uint4*>(in + (int64_t)max(t.y * kCy - 1, 0) * g.X * 32);
    auto load = [&](int z) { stage.load(tile + (int64_t)z * g.sxy * 4, z >= 0 && z < g.Z); };
    float bv[4], hv[4], hb = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        bv[i] = kMode != kBwd ? bias[4 * q + i] : 0.f;
        hv[i] = kMode == kFwdHead ? head[4 * q + i] : 0.f;
    }
    if (kMode == kFwdHead) hb = head[16];
    auto taps = [&](f32x4 acc[kC3Rows], int dz) {
        bf16x8 wt[9];
#pragma unroll
        for (int k = 0; k < 9; k++) wt[k] = load8(wl + (dz * 9 + k) * 512);
#pragma unroll
        for (int i = 0; i < kC3Rows + 2; i++)
#pragma unroll
            for (int dx = 0; dx < 3; dx++) {
                const bf16x8 v = load8(vl + (i * (kCx + 2) + dx) * 32);
#pragma unroll
                for (int dy = 0; dy < 3; dy++)
                    if (i - dy >= 0 && i - dy < kC3Rows)
                        acc[i - dy] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[3 * dy + dx], v, acc[i - dy], 0, 0, 0);
            }
    };
    auto emit = [&](const f32x4 acc[kC3Rows], int z) {
        const int64_t v0 = (int64_t)z * g.sxy + (int64_t)y0 * g.X + x;
        if (kMode == kFwdHead) {
            // head: a vertex's channels are in four lanes; lane q then finishes rows q, q + 4, ..
            float logit[kC3Rows / 4];
#pragma unroll
            for (int j = 0; j < kC3Rows; j++) {
                float p[4];
#pragma unroll
                for (int i = 0; i < 4; i++) p[i] = hv[i] * bf2f((uint16_t)pack_bf(relu(acc[j][i] + bv[i]), 0.f));
                float s = (p[0] + p[1]) + (p[2] + p[3]);
                s += __shfl_xor(s, 16);
                s += __shfl_xor(s, 32);
                if (j % 4 == 0 || q == j % 4) logit[j / 4] = s;
            }
#pragma unroll
            for (int k = 0; k < kC3Rows / 4; k++) {
                const int j = 4 * k + q;
                if (x < g.X && y0 + j < g.Y) prob[v0 + (int64_t)j * g.X] = 1.f / (1.f + expf(-(logit[k] + hb)));
            }
            return;
        }
        if (x >= g.X) return;
#pragma unroll
        for (int j = 0; j < kC3Rows; j++) {
            if (y0 + j >= g.Y) break;
            const int64_t at = (v0 + (int64_t)j * g.X) * 16 + 4 * q;
            uint2 p;
            if (kMode == kFwd) {
                p.x = pack_bf(relu(acc[j][0] + bv[0]), relu(acc[j][1] + bv[1]));
                p.y = pack_bf(relu(acc[j][2] + bv[2]), relu(acc[j][3] + bv[3]));
            } else {
                const uint2 gs = *reinterpret_cast<const uint2*>(gate + at);
                p.x = gated(gs.x, acc[j][0], acc[j][1]);
                p.y = gated(gs.y, acc[j][2], acc[j][3]);
            }
            *reinterpret_cast<uint2*>(out + at) = p;
        }
    };
    f32x4 a[kC3Rows] = {}, b[kC3Rows] = {};  // of the layers below and at the input layer
    load(z0 - 1);
#pragma unroll 1
    for (int z = z0 - 1; z <= z1; z++) {
        __syncthreads();
        stage.store(reinterpret_cast<uint4*>(sv));
        if (z < z1) load(z + 1);
        __syncthreads();
        if (z > z0) {
            taps(a, 2);
            emit(a, z - 1);
        }
        if (z >= z0 && z < z1) {
#pragma unroll
            for (int j = 0; j < kC3Rows; j++) a[j] = b[j];
            taps(a, 1);
        }
        if (z + 1 < z1) {
#pragma unroll
            for (int j = 0; j < kC3Rows; j++) b[j] = f32x4{};
            taps(b, 0);
        }
    }
}

// ---- head + loss (training) -------------------------------------------------

// Per voxel: logit = bh + sum_c wh[c] a3[c], p = sigmoid(logit); weighted BCE
// with weight pos_w on targets 1; dlogit = w (p - t) / n; dz3 = dlogit wh (a3 > 0).
// Per-block partials: [loss, dbh, dwh[16]].
constexpr int kHeadPart = 18;

__global__ void __launch_bounds__(kT)
head_loss_kernel(const uint16_t* __restrict__ a3, Geo g, const float* __restrict__ head, const uint8_t* __restrict__ target,
                 float pos_w, float inv_n, uint16_t* __restrict__ dz3, float* __restrict__ part) {
    __shared__ float red[kT / 64][kHeadPart];
    float acc[kHeadPart] = {};
    float wh[16];
#pragma unroll
    for (int c = 0; c < 16; c++) wh[c] = head[c];
    const float bh = head[16];
    const int64_t n = g.verts();
    for (int64_t v = (int64_t)blockIdx.x * kT + threadIdx.x; v < n; v += (int64_t)gridDim.x * kT) {
        float a[16];
        const uint4* p4 = reinterpret_cast<const uint4*>(a3 + v * 16);
        const uint4 u0 = p4[0], u1 = p4[1];
        const uint32_t w8[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
        for (int c = 0; c < 8; c++) {
            a[2 * c] = bf2f((uint16_t)(w8[c] & 0xFFFFu));
            a[2 * c + 1] = bf2f((uint16_t)(w8[c] >> 16));
        }
        float logit = bh;
#pragma unroll
        for (int c = 0; c < 16; c++) logit = fmaf(wh[c], a[c], logit);
        const float t = target[v] ? 1.f : 0.f;
        const float wgt = target[v] ? pos_w : 1.f;
        // log-sigmoid forms, stable for large |logit|
        const float lsp = logit >= 0.f ? -log1pf(expf(-logit)) : logit - log1pf(expf(logit));  // log p
        const float lsn = lsp - logit;                                                          // log (1-p)
        acc[0] += -wgt * (t * lsp + (1.f - t) * lsn);
        const float p = 1.f / (1.f + expf(-logit));
        const float dl = wgt * (p - t) * inv_n;
        acc[1] += dl;
        uint32_t o[8];
#pragma unroll
        for (int c = 0; c < 16; c += 2) {
            acc[2 + c] += dl * a[c];
            acc[3 + c] += dl * a[c + 1];
            const float d0 = a[c] > 0.f ? dl * wh[c] : 0.f, d1 = a[c + 1] > 0.f ? dl * wh[c + 1] : 0.f;
            o[c / 2] = (uint32_t)f2bf(d0) | ((uint32_t)f2bf(d1) << 16);
        }
        uint4* q4 = reinterpret_cast<uint4*>(dz3 + v * 16);
        q4[0] = make_uint4(o[0], o[1], o[2], o[3]);
        q4[1] = make_uint4(o[4], o[5], o[6], o[7]);
    }
    // block reduction in a fixed order
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < kHeadPart; k++) {
        float x = acc[k];
        for (int m = 32; m >= 1; m >>= 1) x += __shfl_xor(x, m);
        if (lane == 0) red[wave][k] = x;
    }
    __syncthreads();
    if (threadIdx.x < kHeadPart) {
        float x = 0.f;
        for (int w = 0; w < kT / 64; w++) x += red[w][threadIdx.x];
        part[(int64_t)blockIdx.x * kHeadPart + threadIdx.x] = x;
    }
}

// ---- weight gradients (VALU) ------------------------------------------------

// dW[t][co][ci] = sum_v a_in(v + off_t, ci) dz(v, co), db[co] = sum_v dz(v, co).
// A block walks 64-voxel x-segments; the input halo (9 rows x 66 voxels) and
// the gradient segment are staged in LDS.  Thread (co, pair of ci) keeps 27x2
// accumulators; per-block partials [Cout*27*Cin + Cout] are reduced later.
template <int kCin, int kCout>
__global__ void __launch_bounds__(kT)
wgrad_kernel(const uint16_t* __restrict__ ain, const uint16_t* __restrict__ dz, Geo g, float* __restrict__ part) {
    static_assert(kCout * kCin / 2 == kT, "one thread per (co, ci pair)");
    constexpr int kSeg = 64, kW = kSeg + 2;
    __shared__ __attribute__((aligned(16))) uint16_t sa[9 * kW * kCin];
    __shared__ __attribute__((aligned(16))) uint16_t sd[kSeg * kCout];
    const int co = threadIdx.x / (kCin / 2), cp = threadIdx.x % (kCin / 2);
    float acc[27][2] = {};
    float bacc = 0.f;
    const int segs_x = (g.X + kSeg - 1) / kSeg;
    const int64_t nseg = (int64_t)segs_x * g.Y * g.Z;
    for (int64_t sg = blockIdx.x; sg < nseg; sg += gridDim.x) {
        const int x0 = (int)(sg % segs_x) * kSeg;
        const int y = (int)((sg / segs_x) % g.Y), z = (int)(sg / ((int64_t)segs_x * g.Y));
        __syncthreads();
        // stage the input halo: rows (dy, dz), voxels x0-1 .. x0+64, all channels (4-byte words)
        constexpr int kWords = 9 * kW * kCin / 2;
        for (int i = threadIdx.x; i < kWords; i += kT) {
            const int c2 = i % (kCin / 2), rest = i / (kCin / 2);
            const int xi = rest % kW, row = rest / kW;
            const int yy = y + row % 3 - 1, zz = z + row / 3 - 1, xx = x0 - 1 + xi;
            uint32_t val = 0u;
            if (xx >= 0 && xx < g.X && yy >= 0 && yy < g.Y && zz >= 0 && zz < g.Z)
                val = reinterpret_cast<const uint32_t*>(ain + ((int64_t)xx + (int64_t)yy * g.X + (int64_t)zz * g.sxy) * kCin)[c2];
            reinterpret_cast<uint32_t*>(sa)[i] = val;
        }
        for (int i = threadIdx.x; i < kSeg * kCout / 2; i += kT) {
            const int c2 = i % (kCout / 2), xi = i / (kCout / 2), xx = x0 + xi;
            uint32_t val = 0u;
            if (xx < g.X) val = reinterpret_cast<const uint32_t*>(dz + ((int64_t)xx + (int64_t)y * g.X + (int64_t)z * g.sxy) * kCout)[c2];
            reinterpret_cast<uint32_t*>(sd)[i] = val;
        }
        __syncthreads();
        for (int xi = 0; xi < kSeg; xi++) {
            const float d = bf2f(sd[xi * kCout + co]);
            if (d == 0.f) continue;
            bacc += d;
#pragma unroll
            for (int t = 0; t < 27; t++) {
                const int row = (tap_dy(t) + 1) + 3 * (tap_dz(t) + 1);
                const uint32_t pr = reinterpret_cast<const uint32_t*>(sa)[((row * kW) + xi + 1 + tap_dx(t)) * (kCin / 2) + cp];
                acc[t][0] = fmaf(d, bf2f((uint16_t)(pr & 0xFFFFu)), acc[t][0]);
                acc[t][1] = fmaf(d, bf2f((uint16_t)(pr >> 16)), acc[t][1]);
            }
        }
    }
    float* out = part + (int64_t)blockIdx.x * (27 * kCout * kCin + kCout);
#pragma unroll
    for (int t = 0; t < 27; t++) {
        out[(t * kCout + co) * kCin + 2 * cp] = acc[t][0];
        out[(t * kCout + co) * kCin + 2 * cp + 1] = acc[t][1];
    }
    if (cp == 0) out[27 * kCout * kCin + co] = bacc;
}

// conv1 gradient: dW1[t][co] = sum_v n(v + off_t) dz1(v, co), db1[co] = sum_v dz1(v, co).
__global__ void __launch_bounds__(kT)
wgrad1_kernel(const float* __restrict__ xin, const uint16_t* __restrict__ dz1, Geo g, float* __restrict__ part) {
    constexpr int kSeg = 64, kW = kSeg + 2;
    __shared__ float sa[9 * kW];
    __shared__ float sd[kSeg * 16];
    const int co = threadIdx.x % 16, tg = threadIdx.x / 16;  // taps tg and tg + 16
    float acc0 = 0.f, acc1 = 0.f, bacc = 0.f;
    const int segs_x = (g.X + kSeg - 1) / kSeg;
    const int64_t nseg = (int64_t)segs_x * g.Y * g.Z;
    for (int64_t sg = blockIdx.x; sg < nseg; sg += gridDim.x) {
        const int x0 = (int)(sg % segs_x) * kSeg;
        const int y = (int)((sg / segs_x) % g.Y), z = (int)(sg / ((int64_t)segs_x * g.Y));
        __syncthreads();
        for (int i = threadIdx.x; i < 9 * kW; i += kT) {
            const int xi = i % kW, row = i / kW;
            const int yy = y + row % 3 - 1, zz = z + row / 3 - 1, xx = x0 - 1 + xi;
            float val = 0.f;
            if (xx >= 0 && xx < g.X && yy >= 0 && yy < g.Y && zz >= 0 && zz < g.Z)
                val = xin[(int64_t)xx + (int64_t)yy * g.X + (int64_t)zz * g.sxy];
            sa[i] = val;
        }
        for (int i = threadIdx.x; i < kSeg * 16; i += kT) {
            const int c = i % 16, xi = i / 16, xx = x0 + xi;
            sd[i] = xx < g.X ? bf2f(dz1[((int64_t)xx + (int64_t)y * g.X + (int64_t)z * g.sxy) * 16 + c]) : 0.f;
        }
        __syncthreads();
        const int t0 = tg, t1 = tg + 16;
        for (int xi = 0; xi < kSeg; xi++) {
            const float d = sd[xi * 16 + co];
            if (tg == 0) bacc += d;
            {
                const int row = (tap_dy(t0) + 1) + 3 * (tap_dz(t0) + 1);
                acc0 = fmaf(d, sa[row * kW + xi + 1 + tap_dx(t0)], acc0);
            }
            if (t1 < 27) {
                const int row = (tap_dy(t1) + 1) + 3 * (tap_dz(t1) + 1);
                acc1 = fmaf(d, sa[row * kW + xi + 1 + tap_dx(t1)], acc1);
            }
        }
    }
    float* out = part + (int64_t)blockIdx.x * (27 * 16 + 16);
    out[tg * 16 + co] = acc0;
    if (tg + 16 < 27) out[(tg + 16) * 16 + co] = acc1;
    if (tg == 0) out[27 * 16 + co] = bacc;
}

// Sum of per-block partials (fixed order): out[i] = sum_b part[b][i].
__global__ void __launch_bounds__(kT)
reduce_parts_kernel(const float* __restrict__ part, int nblocks, int width, float* __restrict__ out) {
    for (int i = blockIdx.x * kT + threadIdx.x; i < width; i += gridDim.x * kT) {
        double s = 0.0;
        for (int b = 0; b < nblocks; b++) s += (double)part[(int64_t)b * width + i];
        out[i] = (float)s;
    }
}

// [loss, dbh, dwh[16]] -> gradient layout (wh[16], bh at kOffWh)
__global__ void reorder_head_kernel(const float* __restrict__ red, float* __restrict__ grad) {
    const int c = threadIdx.x;
    if (c < 16) grad[kOffWh + c] = red[2 + c];
    if (c == 16) grad[kOffWh + 16] = red[1];
}

// ---- parameters ---------------------------------------------------------------

__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ gr, float* __restrict__ m,
                            float* __restrict__ v, int n, float lr, float b1t, float b2t) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = gr[i];
    const float mi = 0.9f * m[i] + 0.1f * gi;
    const float vi = 0.999f * v[i] + 0.001f * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / (1.f - b1t), vh = vi / (1.f - b2t);
    p[i] -= lr * mh / (sqrtf(vh) + 1e-8f);
}

// Packed operands from the FP32 parameters.
__global__ void pack_kernel(const float* __restrict__ p, CnnPacked k) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kW1) k.w1[i] = bf2f(f2bf(p[kOffW1 + i]));
    if (i < 16) k.b1[i] = p[kOffB1 + i];
    if (i < kW2) {
        // W2 [t][co 32][ci 16] and its mirror-transpose W2T [t'][ci 16][co 32] (t' = 26 - t)
        const uint16_t h = f2bf(p[kOffW2 + i]);
        k.w2[i] = h;
        const int t = i / 512, co = (i / 16) % 32, ci = i % 16;
        k.w2t[((26 - t) * 16 + ci) * 32 + co] = h;
    }
    if (i < 32) k.b2[i] = p[kOffB2 + i];
    if (i < kW3) {
        // W3 [t][co 16][ci 32] and W3T [t'][ci 32][co 16]
        const uint16_t h = f2bf(p[kOffW3 + i]);
        k.w3[i] = h;
        const int t = i / 512, co = (i / 32) % 16, ci = i % 32;
        k.w3t[((26 - t) * 32 + ci) * 16 + co] = h;
    }
    if (i < 16) k.b3[i] = p[kOffB3 + i];
    if (i < 17) k.head[i] = p[kOffWh + i];  // wh[16], bh
}

// ---- mask from probabilities: threshold, then Chebyshev dilation ------------

__global__ void threshold_kernel(const float* __restrict__ prob, int64_t n, float thr, uint8_t* __restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = prob[i] > thr ? 1 : 0;
}

// One axis of a max filter of radius r.
__global__ void dilate_axis_kernel(const uint8_t* __restrict__ in, Geo g, int axis, int r, uint8_t* __restrict__ out) {
    const int64_t n = g.verts();
    const int64_t stride = axis == 0 ? 1 : (axis == 1 ? (int64_t)g.X : g.sxy);
    const int len = axis == 0 ? g.X : (axis == 1 ? g.Y : g.Z);
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x) {
        const int c = axis == 0 ? (int)(v % g.X) : (axis == 1 ? (int)((v / g.X) % g.Y) : (int)(v / g.sxy));
        uint8_t m = 0;
        for (int d = -r; d <= r; d++) {
            const int cc = c + d;
            if (cc < 0 || cc >= len) continue;
            m |= in[v + d * stride];
        }
        out[v] = m;
    }
}

__global__ void count_kernel(const uint8_t* __restrict__ m, int64_t n, unsigned long long* __restrict__ out) {
    uint32_t c = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        c += m[i] ? 1u : 0u;
    for (int s = 32; s >= 1; s >>= 1) c += __shfl_xor(c, s);
    if ((threadIdx.x & 63) == 0 && c) atomicAdd(out, (unsigned long long)c);
}

// launch(grid, tiles) for all x * y * z tiles of the volume (fewer than 2^30: a
// volume has at most 2^34 vertices and sides of 2^16, a tile 4 rows or more).
template <class Launch>
void for_tiles(const Geo& g, int x, int y, int z, Launch launch) {
    auto along = [](int n, int side) { return (uint32_t)((n + side - 1) / side); };
    Tiles t{0, 0, along(g.X, x), along(g.Y, y)};
    const uint32_t all = t.x * t.y * along(g.Z, z);
    for (; t.first < all; t.first += t.n) {
        t.n = std::min(all - t.first, kMaxTiles);
        launch(dim3(t.n), t);
    }
}
// Layers a work-group of a convolution runs up: the more, the fewer layers are
// read twice and the fewer weights staged, as long as there are two work-groups
// per CU.
inline int conv_layers(const Geo& g) {
    const int64_t tiles = (int64_t)((g.X + kCx - 1) / kCx) * ((g.Y + kCy - 1) / kCy);
    int n = 8;
    while (n > 1 && tiles * ((g.Z + n - 1) / n) < 512) n /= 2;
    return n;
}
inline uint32_t blocks_for(int64_t n, uint32_t cap = 16384) {
    const int64_t b = (n + kT - 1) / kT;
    return (uint32_t)(b < 1 ? 1 : (b > cap ? cap : b));
}

// SplitMix64 -> uniform (0,1) -> normal (Box-Muller), for the initial weights.
struct Rng {
    uint64_t s;
    uint64_t next() {
        uint64_t z = (s += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    }
    double uniform() { return ((double)(next() >> 11) + 0.5) * (1.0 / 9007199254740992.0); }
    double normal() {
        const double u1 = uniform(), u2 = uniform();
        return std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
    }
};

}  // namespace

// ---- host side -----------------------------------------------------------------

std::vector<float> cnn_initial_params(uint64_t seed) {
    std::vector<float> p(kNumParams, 0.f);
    Rng rng{seed};
    auto he = [&](int off, int n, int fan_in) {
        const double s = std::sqrt(2.0 / fan_in);
        for (int i = 0; i < n; i++) p[off + i] = (float)(s * rng.normal());
    };
    he(kOffW1, kW1, 27);
    he(kOffW2, kW2, 27 * 16);
    he(kOffW3, kW3, 27 * 32);
    for (int i = 0; i < 16; i++) p[kOffWh + i] = (float)(std::sqrt(1.0 / 16) * rng.normal());
    p[kOffWh + 16] = -1.0f;  // start below 0.5: most voxels are negatives
    return p;
}

hipError_t CnnState::ensure_volume(int64_t verts) {
    if (verts <= vol_cap) return hipSuccess;
    hipError_t e;
    if ((e = tmp.ensure(sizeof(double2) * verts)) != hipSuccess) return e;
    if ((e = xin.ensure(sizeof(float) * verts)) != hipSuccess) return e;
    if ((e = a1.ensure(2 * 16 * verts)) != hipSuccess) return e;
    if ((e = a2.ensure(2 * 32 * verts)) != hipSuccess) return e;
    if ((e = a3.ensure(2 * 16 * verts)) != hipSuccess) return e;
    if ((e = prob.ensure(sizeof(float) * verts)) != hipSuccess) return e;
    if ((e = m0.ensure(verts)) != hipSuccess) return e;
    if ((e = m1.ensure(verts)) != hipSuccess) return e;
    vol_cap = verts;
    return hipSuccess;
}

hipError_t CnnState::ensure_train(int64_t verts) {
    hipError_t e;
    if ((e = dz3.ensure(2 * 16 * verts)) != hipSuccess) return e;
    if ((e = dz2.ensure(2 * 32 * verts)) != hipSuccess) return e;
    if ((e = dz1.ensure(2 * 16 * verts)) != hipSuccess) return e;
    return hipSuccess;
}

void CnnState::release_all() {
    DevBuf* all[] = {&params, &grads, &m, &v, &pk, &parts, &loss, &tmp, &xin, &a1, &a2, &a3,
                     &prob, &m0, &m1, &dz3, &dz2, &dz1};
    for (DevBuf* b : all) b->release();
    vol_cap = 0;
}

CnnPacked CnnState::packed() const {
    CnnPacked k;
    uint8_t* base = pk.as<uint8_t>();
    k.w1 = reinterpret_cast<float*>(base);
    k.b1 = k.w1 + kW1;
    k.b2 = k.b1 + 16;
    k.b3 = k.b2 + 32;
    k.head = k.b3 + 16;
    uint16_t* h = reinterpret_cast<uint16_t*>(base + 4096);
    k.w2 = h;
    k.w2t = h + kW2;
    k.w3 = h + 2 * kW2;
    k.w3t = h + 2 * kW2 + kW3;
    return k;
}

hipError_t cnn_pack(CnnState& s, hipStream_t st) {
    hipLaunchKernelGGL(pack_kernel, dim3((kW2 + kT - 1) / kT), dim3(kT), 0, st, s.params.as<float>(), s.packed());
    return hipGetLastError();
}

hipError_t cnn_forward(CnnState& s, const float* values, int X, int Y, int Z, bool keep_a3, float* prob, hipStream_t st) {
    const Geo g{X, Y, Z, (int64_t)X * Y};
    const CnnPacked k = s.packed();
    const int layers = conv_layers(g);
    for_tiles(g, kNormX, kNormY, 1, [&](dim3 n, Tiles t) {
        hipLaunchKernelGGL(norm_xy_kernel, n, dim3(kT), 0, st, values, g, t, s.tmp.as<double2>());
    });
    for_tiles(g, 64, kT / 64, kNormZ, [&](dim3 n, Tiles t) {
        hipLaunchKernelGGL(norm_z_kernel, n, dim3(kT), 0, st, s.tmp.as<double2>(), values, g, t, s.xin.as<float>());
    });
    for_tiles(g, 64, kC1Rows, kT / 64, [&](dim3 n, Tiles t) {
        hipLaunchKernelGGL(conv1_kernel, n, dim3(kT), 0, st, s.xin.as<float>(), g, t, k.w1, k.b1, s.a1.as<uint16_t>());
    });
    for_tiles(g, kCx, kCy, layers, [&](dim3 n, Tiles t) {
        hipLaunchKernelGGL(conv16to32_kernel<kFwd>, n, dim3(kT), 0, st, s.a1.as<uint16_t>(), g, t, layers, k.w2, k.b2,
                           (const uint16_t*)nullptr, s.a2.as<uint16_t>());
    });
    for_tiles(g, kCx, kCy, layers, [&](dim3 n, Tiles t) {
        if (keep_a3)
            hipLaunchKernelGGL(conv32to16_kernel<kFwd>, n, dim3(kT), 0, st, s.a2.as<uint16_t>(), g, t, layers, k.w3, k.b3, k.head,
                               (const uint16_t*)nullptr, s.a3.as<uint16_t>(), (float*)nullptr);
        else
            hipLaunchKernelGGL(conv32to16_kernel<kFwdHead>, n, dim3(kT), 0, st, s.a2.as<uint16_t>(), g, t, layers, k.w3, k.b3,
                               k.head, (const uint16_t*)nullptr, (uint16_t*)nullptr, prob);
    });
    return hipGetLastError();
}

hipError_t cnn_backward(CnnState& s, int X, int Y, int Z, const uint8_t* target, float pos_w, hipStream_t st) {
    const Geo g{X, Y, Z, (int64_t)X * Y};
    const int64_t n = g.verts();
    const CnnPacked k = s.packed();
    const uint32_t hb = blocks_for(n, 1024);
    hipLaunchKernelGGL(head_loss_kernel, dim3(hb), dim3(kT), 0, st, s.a3.as<uint16_t>(), g, k.head, target, pos_w,
                       (float)(1.0 / (double)n), s.dz3.as<uint16_t>(), s.parts.as<float>());
    float* grad = s.grads.as<float>();
    float* loss = s.loss.as<float>();
    // head: [loss, dbh, dwh[16]] -> loss, grads at kOffWh
    hipLaunchKernelGGL(reduce_parts_kernel, dim3(1), dim3(kT), 0, st, s.parts.as<float>(), (int)hb, kHeadPart,
                       loss);
    hipLaunchKernelGGL(reorder_head_kernel, dim3(1), dim3(32), 0, st, loss, grad);
    // dz2 = (dz3 conv^T W3) * (a2 > 0): a 16 -> 32 convolution with W3T
    const int layers = conv_layers(g);
    for_tiles(g, kCx, kCy, layers, [&](dim3 n, Tiles t) {
        hipLaunchKernelGGL(conv16to32_kernel<kBwd>, n, dim3(kT), 0, st, s.dz3.as<uint16_t>(), g, t, layers, k.w3t,
                           (const float*)nullptr, s.a2.as<uint16_t>(), s.dz2.as<uint16_t>());
    });
    // dz1 = (dz2 conv^T W2) * (a1 > 0): a 32 -> 16 convolution with W2T
    for_tiles(g, kCx, kCy, layers, [&](dim3 n, Tiles t) {
        hipLaunchKernelGGL(conv32to16_kernel<kBwd>, n, dim3(kT), 0, st, s.dz2.as<uint16_t>(), g, t, layers, k.w2t,
                           (const float*)nullptr, (const float*)nullptr, s.a1.as<uint16_t>(), s.dz1.as<uint16_t>(),
                           (float*)nullptr);
    });
    const int64_t nseg = (int64_t)((X + 63) / 64) * Y * Z;
    const int wb = (int)std::min<int64_t>(nseg, kGradBlocks);
    hipLaunchKernelGGL((wgrad_kernel<32, 16>), dim3(wb), dim3(kT), 0, st, s.a2.as<uint16_t>(), s.dz3.as<uint16_t>(), g,
                       s.parts.as<float>());
    hipLaunchKernelGGL(reduce_parts_kernel, dim3((kW3 + 16 + kT - 1) / kT), dim3(kT), 0, st, s.parts.as<float>(), wb,
                       kW3 + 16, grad + kOffW3);
    hipLaunchKernelGGL((wgrad_kernel<16, 32>), dim3(wb), dim3(kT), 0, st, s.a1.as<uint16_t>(), s.dz2.as<uint16_t>(), g,
                       s.parts.as<float>());
    hipLaunchKernelGGL(reduce_parts_kernel, dim3((kW2 + 32 + kT - 1) / kT), dim3(kT), 0, st, s.parts.as<float>(), wb,
                       kW2 + 32, grad + kOffW2);
    hipLaunchKernelGGL(wgrad1_kernel, dim3(wb), dim3(kT), 0, st, s.xin.as<float>(), s.dz1.as<uint16_t>(), g,
                       s.parts.as<float>());
    hipLaunchKernelGGL(reduce_parts_kernel, dim3((kW1 + 16 + kT - 1) / kT), dim3(kT), 0, st, s.parts.as<float>(), wb,
                       kW1 + 16, grad + kOffW1);
    return hipGetLastError();
}

hipError_t cnn_adam(CnnState& s, float lr, hipStream_t st) {
    s.step++;
    const float b1t = std::pow(0.9f, (float)s.step), b2t = std::pow(0.999f, (float)s.step);
    hipLaunchKernelGGL(adam_kernel, dim3((kNumParams + kT - 1) / kT), dim3(kT), 0, st, s.params.as<float>(),
                       s.grads.as<float>(), s.m.as<float>(), s.v.as<float>(), kNumParams, lr, b1t, b2t);
    return cnn_pack(s, st);
}

hipError_t cnn_mask(CnnState& s, int X, int Y, int Z, float thr, int dilation, uint8_t* out,
                    unsigned long long* count, hipStream_t st) {
    const Geo g{X, Y, Z, (int64_t)X * Y};
    const int64_t n = g.verts();
    uint8_t* a = dilation > 0 ? s.m0.as<uint8_t>() : out;
    hipLaunchKernelGGL(threshold_kernel, dim3(blocks_for(n)), dim3(kT), 0, st, s.prob.as<float>(), n, thr, a);
    if (dilation > 0) {
        hipLaunchKernelGGL(dilate_axis_kernel, dim3(blocks_for(n)), dim3(kT), 0, st, s.m0.as<uint8_t>(), g, 0, dilation,
                           s.m1.as<uint8_t>());
        hipLaunchKernelGGL(dilate_axis_kernel, dim3(blocks_for(n)), dim3(kT), 0, st, s.m1.as<uint8_t>(), g, 1, dilation,
                           s.m0.as<uint8_t>());
        hipLaunchKernelGGL(dilate_axis_kernel, dim3(blocks_for(n)), dim3(kT), 0, st, s.m0.as<uint8_t>(), g, 2, dilation,
                           out);
    }
    if (count) hipLaunchKernelGGL(count_kernel, dim3(blocks_for(n, 4096)), dim3(kT), 0, st, out, n, count);
    return hipGetLastError();
}

}  // namespace msceer
