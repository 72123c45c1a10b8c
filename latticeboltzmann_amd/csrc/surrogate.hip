// Kernels of the warm-start surrogate: a small convolutional encoder-decoder
// trained and evaluated on the GPU, plus the initializer that turns its
// prediction into populations.
//
// Convolutions are 3x3, stride 1, zero padding, NHWC activations: products of the
// neighbourhoods cols[pixel][(dy*3+dx)*C + c] (BF16) with the weights
// W[cout][(dy*3+dx)*C + c] (BF16), accumulated in FP32 by v_mfma_f32_16x16x32_bf16
// (gfx950).  k_conv3p (packed weights) and k_conv3 do the forward pass and the
// data gradient where the input channels are a multiple of 32, k_wgrad the weight
// gradient (split over pixels, the splits added in order), k_gemm with its
// gathering loaders the rest; no atomics, so every result is deterministic.
// For training, activations are kept in FP32 with a BF16 copy for the next
// product; weights in FP32 (Adam) with a BF16 copy.
//
// No reference counterpart: the reference has no learned component.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <initializer_list>

#include "d2q9_node.hpp"
#include "d2q9_reduce.hpp"
#include "lbm_internal.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace lbm {
namespace nn {

__device__ __forceinline__ float bf2f(uint16_t x) { return float(__builtin_bit_cast(__bf16, x)); }
__device__ __forceinline__ uint16_t f2bf(float x) { return __builtin_bit_cast(uint16_t, __bf16(x)); }

// ---------------------------------------------------------------------------
// GEMM: C[m][n] = sum_k A(m, k) B(k, n), A(m, k) = A[m*sam + k*sak],
// B(k, n) = B[k*sbk + n*sbn] (BF16), FP32 accumulation.
// Block: 256 threads = 4 waves, tile 64 x 64, k-step 32 staged in LDS as
// As[m][k] and Bs[n][k]; each wave owns a 32 x 32 quarter = 2 x 2 MFMA
// 16x16x32 tiles, and reads each operand as 8 consecutive k of one row.
// MFMA operand layout (checked on gfx950): lane l holds A rows l%16,
// k = (l/16)*8 + i; B cols l%16, k = (l/16)*8 + i; result register r of lane l
// is row (l/16)*4 + r, col l%16.
// Tile loads (per operand, chosen on the host): LOAD_K: k contiguous, each
// thread loads 8 k of one row with one 16-byte load; LOAD_ROW: the row index
// contiguous, each thread loads 8 rows of one k; LOAD_SCALAR otherwise.  The
// vector forms need 16-byte alignment of the base and of the other stride
// and fall back to bounds-checked scalar loads at partial tiles.
// Split-K: blockIdx.z handles k in [z*kchunk, (z+1)*kchunk); with more than
// one split, results go to work[z][m][n] and k_gemm_reduce adds them in order.
constexpr int TM = 64, TN = 64, TK = 32, TP = TK + 8;
constexpr int LOAD_SCALAR = 0, LOAD_K = 1, LOAD_ROW = 2;

// A convolution operand gathered on the fly instead of read from a
// materialised im2col matrix: element (pixel p, index q) with q = tap * C + c,
// tap = (dy + 1) * 3 + (dx + 1), is X[pixel p + sign * (dy, dx)][c] of the NHWC
// BF16 activation X (H x W images, C channels), 0 outside the image.  sign +1
// is the im2col of a 3x3 same convolution; sign -1 gathers, for input pixel
// p, the output pixels that read p (the data gradient).  sign 0: no gather.
struct Gather {
    int H, W, C, sign;
};

struct GemmArgs {
    const uint16_t *A;
    int64_t sam, sak;
    const uint16_t *B;
    int64_t sbk, sbn;
    float *C;      // FP32 output (nullable)
    uint16_t *Cb;  // BF16 output (nullable)
    int64_t ldc;
    const float *bias;
    int M, N, K, kchunk, accumulate, relu;
    float *work;   // split-K partials
    int mode_a, mode_b;
    Gather ga;     // A(m, k) gathered with pixel m, index k (ga.sign != 0)
    Gather gb;     // B(k, n) gathered with pixel k, index n (gb.sign != 0)
};

// Index into X of gathered element (pixel p, index q), and whether it lies in
// the image.
__device__ __forceinline__ int64_t gather_index(const Gather &G, int p, int q, bool &inside) {
    const int tap = q / G.C, c = q - tap * G.C;
    const int dy = (tap / 3 - 1) * G.sign, dx = (tap % 3 - 1) * G.sign;
    const int x = p % G.W, y = (p / G.W) % G.H;
    inside = unsigned(y + dy) < unsigned(G.H) && unsigned(x + dx) < unsigned(G.W);
    return (int64_t(p) + int64_t(dy) * G.W + dx) * G.C + c;
}

__device__ __forceinline__ uint16_t gather_one(const uint16_t *__restrict__ X, const Gather &G,
                                               int p, int q) {
    bool in;
    const int64_t i = gather_index(G, p, q, in);
    return in ? X[i] : uint16_t(0);
}

// tile[row][k] <- X(row0 + row, k0 + k) for a gathered operand, zero outside
// rows < nrows, k < kend.  pix_row: the row is the pixel and k the (tap,
// channel) index (A of the forward and data-gradient GEMMs); otherwise k is
// the pixel and the row the index (B of the weight-gradient GEMM).  With C a
// multiple of 8, the 8 indices a thread loads lie in one tap: one 16-byte load.
__device__ __forceinline__ void load_tile_gather(uint16_t (*tile)[TP], const uint16_t *__restrict__ X,
                                                 const Gather &G, int row0, int nrows, int k0,
                                                 int kend, bool pix_row, int t) {
    const bool vec = G.C % 8 == 0;
    if (pix_row) {
        const int rr = t >> 2, kc = (t & 3) * 8;
        const int r = row0 + rr, k = k0 + kc;
        if (vec && r < nrows && k + 8 <= kend) {
            bool in;
            const int64_t i = gather_index(G, r, k, in);
            uint4 v = make_uint4(0, 0, 0, 0);
            if (in) v = *reinterpret_cast<const uint4 *>(X + i);
            *reinterpret_cast<uint4 *>(&tile[rr][kc]) = v;
            return;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            tile[rr][kc + i] = (r < nrows && k + i < kend) ? gather_one(X, G, r, k + i) : uint16_t(0);
        return;
    }
    const int kr = t >> 3, rc = (t & 7) * 8;
    const int k = k0 + kr, r = row0 + rc;
    if (vec && k < kend && r + 8 <= nrows) {
        bool in;
        const int64_t i = gather_index(G, k, r, in);
        uint4 v = make_uint4(0, 0, 0, 0);
        if (in) v = *reinterpret_cast<const uint4 *>(X + i);
        const uint16_t *e = reinterpret_cast<const uint16_t *>(&v);
#pragma unroll
        for (int i = 0; i < 8; ++i) tile[rc + i][kr] = e[i];
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
        tile[rc + i][kr] = (k < kend && r + i < nrows) ? gather_one(X, G, k, r + i) : uint16_t(0);
}

// tile[row][k] <- X(row0 + row, k0 + k) for row < 64, k < 32; X(r, k) =
// X[r*s_row + k*s_k], zero outside rows < nrows, k < kend.
__device__ __forceinline__ void load_tile(uint16_t (*tile)[TP], const uint16_t *__restrict__ X,
                                          int64_t s_row, int64_t s_k, int row0, int nrows, int k0,
                                          int kend, int mode, int t) {
    if (mode == LOAD_ROW) {
        const int kr = t >> 3, rc = (t & 7) * 8;
        const int k = k0 + kr, r = row0 + rc;
        if (k < kend && r + 8 <= nrows) {
            const uint4 v = *reinterpret_cast<const uint4 *>(X + int64_t(k) * s_k + r);
            const uint16_t *e = reinterpret_cast<const uint16_t *>(&v);
#pragma unroll
            for (int i = 0; i < 8; ++i) tile[rc + i][kr] = e[i];
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                tile[rc + i][kr] = (k < kend && r + i < nrows) ? X[int64_t(k) * s_k + r + i] : 0;
        }
        return;
    }
    const int rr = t >> 2, kc = (t & 3) * 8;
    const int r = row0 + rr, k = k0 + kc;
    if (mode == LOAD_K && r < nrows && k + 8 <= kend) {
        *reinterpret_cast<uint4 *>(&tile[rr][kc]) =
            *reinterpret_cast<const uint4 *>(X + int64_t(r) * s_row + k);
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
        tile[rr][kc + i] = (r < nrows && k + i < kend) ? X[int64_t(r) * s_row + int64_t(k + i) * s_k] : 0;
}

__global__ __launch_bounds__(256) void k_gemm(GemmArgs g) {
    __shared__ __align__(16) uint16_t As[TM][TP];
    __shared__ __align__(16) uint16_t Bs[TN][TP];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    const int kbeg = blockIdx.z * g.kchunk;
    const int kend = min(g.K, kbeg + g.kchunk);
    const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
    floatx4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    for (int k0 = kbeg; k0 < kend; k0 += TK) {
        if (g.ga.sign) load_tile_gather(As, g.A, g.ga, m0, g.M, k0, kend, true, t);
        else load_tile(As, g.A, g.sam, g.sak, m0, g.M, k0, kend, g.mode_a, t);
        if (g.gb.sign) load_tile_gather(Bs, g.B, g.gb, n0, g.N, k0, kend, false, t);
        else load_tile(Bs, g.B, g.sbn, g.sbk, n0, g.N, k0, kend, g.mode_b, t);
        __syncthreads();
        bf16x8 a[2], b[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
            a[i] = *reinterpret_cast<const bf16x8 *>(&As[wm + i * 16 + (lane & 15)][(lane >> 4) * 8]);
#pragma unroll
        for (int j = 0; j < 2; ++j)
            b[j] = *reinterpret_cast<const bf16x8 *>(&Bs[wn + j * 16 + (lane & 15)][(lane >> 4) * 8]);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        __syncthreads();
    }

    const bool split = gridDim.z > 1;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + wm + i * 16 + (lane >> 4) * 4 + r;
                const int n = n0 + wn + j * 16 + (lane & 15);
                if (m >= g.M || n >= g.N) continue;
                float v = acc[i][j][r];
                if (split) {
                    g.work[(int64_t(blockIdx.z) * g.M + m) * g.N + n] = v;
                    continue;
                }
                const int64_t o = int64_t(m) * g.ldc + n;
                if (g.accumulate) v += g.C[o];
                if (g.bias) v += g.bias[n];
                if (g.relu) v = fmaxf(v, 0.0f);
                if (g.C) g.C[o] = v;
                if (g.Cb) g.Cb[o] = f2bf(v);
            }
}

// Fixed-order sum of the split-K partials plus the epilogue.
__global__ __launch_bounds__(256) void k_gemm_reduce(GemmArgs g, int splits) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= int64_t(g.M) * g.N) return;
    const int m = int(idx / g.N), n = int(idx - int64_t(m) * g.N);
    float v = 0.0f;
    for (int z = 0; z < splits; ++z) v += g.work[int64_t(z) * g.M * g.N + idx];
    const int64_t o = int64_t(m) * g.ldc + n;
    if (g.accumulate) v += g.C[o];
    if (g.bias) v += g.bias[n];
    if (g.relu) v = fmaxf(v, 0.0f);
    if (g.C) g.C[o] = v;
    if (g.Cb) g.Cb[o] = f2bf(v);
}

// ---------------------------------------------------------------------------
// 3x3 same convolution with C % 32 == 0 input channels: out[p][n] = sum over
// taps and c of X[p + sign * tap][c] W[n][tap * C + c], NHWC BF16, FP32
// accumulation in the k order of k_gemm (tap by tap, 32 channels a step), so
// the results are its bits.  sign +1: forward; -1: data gradient.
//
// Both MFMA operands want 8 consecutive channels of one row per lane, which is
// how X and W lie in memory, so every lane loads its fragments straight into
// registers (16 bytes each): no LDS, no barrier, D steps of loads in flight per
// wave.  (k_gemm moves each step's tiles through LDS between two barriers with
// nothing in flight: about 1 us per step, whatever the step computes.)  Pixels
// outside the image are loaded from an offset past the buffer's end, which the
// buffer load answers with zeros.  The weights are the MFMA's row operand, so a
// lane ends with 4 consecutive output channels of one pixel: 16-byte stores.
// A wave computes MT x 16 pixels x NT x 16 channels; the 4 waves of a block
// take consecutive pixels and share the weights through L1.
struct ConvArgs {
    const uint16_t *X, *Wt;
    float *y;      // nullable
    uint16_t *yb;  // nullable
    const float *bias;
    int P, H, W, C, N, sign, accumulate, relu;
};

// Stores 4 consecutive output channels c of pixel p.
__device__ __forceinline__ void conv_store(const ConvArgs &a, floatx4 v, int p, int c) {
    if (p >= a.P) return;
    const int64_t o = int64_t(p) * a.N + c;
    if ((a.N & 3) == 0) {
        if (c >= a.N) return;
        if (a.accumulate) v += *reinterpret_cast<const floatx4 *>(a.y + o);
        if (a.bias) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += a.bias[c + r];
        }
        if (a.relu) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = fmaxf(v[r], 0.0f);
        }
        if (a.y) *reinterpret_cast<floatx4 *>(a.y + o) = v;
        if (a.yb)
            *reinterpret_cast<ushort4 *>(a.yb + o) = make_ushort4(f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3]));
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (c + r >= a.N) continue;
        float u = v[r];
        if (a.accumulate) u += a.y[o + r];
        if (a.bias) u += a.bias[c + r];
        if (a.relu) u = fmaxf(u, 0.0f);
        if (a.y) a.y[o + r] = u;
        if (a.yb) a.yb[o + r] = f2bf(u);
    }
}

template <int MT, int NT, int D>
__global__ __launch_bounds__(256) void k_conv3(ConvArgs a) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(int(blockIdx.x * 4 + (threadIdx.x >> 6)));
    const int p0 = wave * 16 * MT, n0 = blockIdx.y * 16 * NT;
    if (p0 >= a.P) return;
    const int col = lane & 15, kq = (lane >> 4) * 8;
    const unsigned xbytes = unsigned(a.P) * unsigned(a.C) * 2u;
    const unsigned wbytes = unsigned(a.N) * 9u * unsigned(a.C) * 2u;
    __amdgpu_buffer_rsrc_t xr =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(a.X), 0, int(xbytes), 0x00020000);
    __amdgpu_buffer_rsrc_t wr =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(a.Wt), 0, int(wbytes), 0x00020000);
    constexpr unsigned kOutside = 0x80000000u;  // past any operand (host: below 2^31 bytes)

    unsigned xo[MT];   // byte offset of the lane's pixel
    unsigned in[MT];   // bit `tap`: the tap's pixel lies in the image
    unsigned wo[NT];   // byte offset of the lane's weight row
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int p = p0 + m * 16 + col;
        const int x = p % a.W, y = (p / a.W) % a.H;
        unsigned bits = 0;
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            const int yy = y + a.sign * (tap / 3 - 1), xx = x + a.sign * (tap % 3 - 1);
            bits |= unsigned(p < a.P && unsigned(yy) < unsigned(a.H) && unsigned(xx) < unsigned(a.W)) << tap;
        }
        in[m] = bits;
        xo[m] = (unsigned(p) * unsigned(a.C) + unsigned(kq)) * 2u;
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int r = n0 + n * 16 + col;
        wo[n] = r < a.N ? (unsigned(r) * 9u * unsigned(a.C) + unsigned(kq)) * 2u : kOutside;
    }

    floatx4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = floatx4{0.f, 0.f, 0.f, 0.f};

    const int per_tap = a.C / 32, S = 9 * per_tap;  // S is a multiple of D
    u32x4 fx[D][MT], fw[D][NT];
    int tap = 0, cc = 0, step = 0;  // of the next load
    auto load = [&](u32x4 *bx, u32x4 *bw) {
        const int shift = a.sign * ((tap / 3 - 1) * a.W + (tap % 3 - 1)) * a.C * 2 + cc * 64;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const unsigned o = (in[m] >> tap) & 1u ? xo[m] + unsigned(shift) : kOutside;
            bx[m] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, int(o), 0, 0));
        }
#pragma unroll
        for (int n = 0; n < NT; ++n)
            bw[n] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                  wr, int(wo[n]), step * 64, 0));
        ++step;
        if (++cc == per_tap) cc = 0, ++tap;
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load(fx[d], fw[d]);
    for (int s = 0; s < S; s += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, fw[d][n]), __builtin_bit_cast(bf16x8, fx[d][m]),
                        acc[m][n], 0, 0, 0);
            if (s + D < S) load(fx[d], fw[d]);
        }
    }

#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
            conv_store(a, acc[m][n], p0 + m * 16 + col, n0 + n * 16 + (lane >> 4) * 4);
}

// The same convolution for the network's own calls: the pixels a block's taps
// read, one run of the flattened image, are staged in LDS once (rows of C
// channels padded by 16 bytes, so the 16 rows of a fragment fall into different
// banks), and the weights come packed in fragment order (k_pack_weights), 1 KB
// of consecutive bytes a load.  k_conv3 is bound by its loads' addresses, 16
// rows a load (some 80 cycles of a CU each, L1 hit or not); here only the staging
// has rows to address.  Row 0 of the LDS holds zeros for pixels outside the image.
// Waves 2 x 2: pixels 32 MT, channels 32 NT a block.
template <int MT, int NT, int D>
__global__ __launch_bounds__(256) void k_conv3p(ConvArgs a) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    extern __shared__ __align__(16) unsigned char smem[];
    const int t = threadIdx.x, lane = t & 63, col = lane & 15, kq = (lane >> 4) * 8;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6), wm = w >> 1, wn = w & 1;
    const int pitch = a.C * 2 + 16;
    const int pb = blockIdx.x * 32 * MT, r0 = pb - a.W - 1;  // pixel of LDS row 1
    __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(a.X), 0, int(unsigned(a.P) * unsigned(a.C) * 2u), 0x00020000);
    const int S = 9 * (a.C / 32), per_tap = a.C / 32;
    __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(a.Wt), 0, (a.N + 15) / 16 * S * 1024, 0x00020000);

    u32x4 fw[D][NT];
    unsigned wo[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) wo[n] = unsigned(((blockIdx.y * 2 + wn) * NT + n) * S * 1024 + lane * 16);
    auto load_w = [&](u32x4 *bw, int step) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
            bw[n] = __builtin_bit_cast(
                u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, int(wo[n] + unsigned(step) * 1024u), 0, 0));
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load_w(fw[d], d);

    {
        const int cpr = a.C / 8, items = (32 * MT + 2 * a.W + 2) * cpr;
        const float inv = 1.0f / float(cpr);
        if (t * 16 < pitch) *reinterpret_cast<u32x4 *>(smem + t * 16) = u32x4{0, 0, 0, 0};
#pragma unroll 4
        for (int i = t; i < items; i += 256) {
            const int r = int((float(i) + 0.5f) * inv), c = i - r * cpr;
            const int q = r0 + r;
            const unsigned o = q >= 0 && q < a.P ? unsigned(q) * unsigned(a.C) * 2u + unsigned(c) * 16u : 0x80000000u;
            *reinterpret_cast<u32x4 *>(smem + (r + 1) * pitch + c * 16) =
                __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, int(o), 0, 0));
        }
    }

    unsigned in[MT];
    int base[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int lp = (wm * MT + m) * 16 + col, p = pb + lp;
        const int x = p % a.W, y = (p / a.W) % a.H;
        unsigned bits = 0;
#pragma unroll
        for (int tap = 0; tap < 9; ++tap) {
            const int yy = y + a.sign * (tap / 3 - 1), xx = x + a.sign * (tap % 3 - 1);
            bits |= unsigned(p < a.P && unsigned(yy) < unsigned(a.H) && unsigned(xx) < unsigned(a.W)) << tap;
        }
        in[m] = bits;
        base[m] = (lp + a.W + 2) * pitch + kq * 2;
    }
    floatx4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = floatx4{0.f, 0.f, 0.f, 0.f};
    __syncthreads();

    int tap = 0, cc = 0, at[MT];
    for (int s = 0; s < S; s += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (cc == 0) {
                const int shift = a.sign * ((tap / 3 - 1) * a.W + (tap % 3 - 1)) * pitch;
#pragma unroll
                for (int m = 0; m < MT; ++m) at[m] = (in[m] >> tap) & 1u ? base[m] + shift : kq * 2;
            }
            bf16x8 x[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) x[m] = *reinterpret_cast<const bf16x8 *>(smem + at[m] + cc * 64);
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fw[d][n]), x[m],
                                                                        acc[m][n], 0, 0, 0);
            if (s + D + d < S) load_w(fw[d], s + D + d);
            if (++cc == per_tap) cc = 0, ++tap;
        }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
            conv_store(a, acc[m][n], pb + (wm * MT + m) * 16 + col,
                       ((blockIdx.y * 2 + wn) * NT + n) * 16 + (lane >> 4) * 4);
}

// Weights of several layers in the fragment order of k_conv3p: for output channel
// tile i and 32-channel step s, lane l holds channels k = 32 s + (l / 16) 8 .. + 7 of
// output i 16 + l % 16 (zero past the last).  forward: output co, k = tap cin + c;
// transposed (the data gradient): output c, k = tap cout + co.
struct PackTable {
    int n, transposed;
    int64_t from[LBM_NN_MAX_LAYERS], to[LBM_NN_MAX_LAYERS];  // elements
    int cin[LBM_NN_MAX_LAYERS], cout[LBM_NN_MAX_LAYERS], first[LBM_NN_MAX_LAYERS + 1];
};

__global__ __launch_bounds__(256) void k_pack_weights(const uint16_t *__restrict__ w, uint16_t *__restrict__ out,
                                                      const PackTable q) {
    int j = 0;
    while (int(blockIdx.x) >= q.first[j + 1]) ++j;
    const int cin = q.cin[j], cout = q.cout[j];
    const int K = q.transposed ? cout : cin, N = q.transposed ? cin : cout, S = 9 * K / 32;
    const int i = (int(blockIdx.x) - q.first[j]) * 256 + int(threadIdx.x);  // (tile, step, lane)
    if (i >= (N + 15) / 16 * S * 64) return;
    const int lane = i & 63, s = (i >> 6) % S, n = (i >> 6) / S * 16 + (lane & 15);
    const int k = s * 32 + (lane >> 4) * 8, tap = k / K, c = k - tap * K;
    const uint16_t *src = w + q.from[j];
    uint16_t v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        v[e] = 0;
        if (n < N) v[e] = q.transposed ? src[(int64_t(c + e) * 9 + tap) * cin + n] : src[(int64_t(n) * 9 + tap) * cin + c + e];
    }
    uint4 o = make_uint4(v[0] | unsigned(v[1]) << 16, v[2] | unsigned(v[3]) << 16, v[4] | unsigned(v[5]) << 16,
                         v[6] | unsigned(v[7]) << 16);
    *reinterpret_cast<uint4 *>(out + q.to[j] + int64_t(i) * 8) = o;
}

// Weight gradient of the 3x3 convolution: dW[co][tap * C + c] = sum over pixels
// of dY[p][co] X[p + tap][c].  Here the MFMA's k is the pixel, and both operands
// lie channel by channel, so a block stages 128 pixels at a time in LDS with
// pixels and channels exchanged: a thread loads 8 pixels x 8 channels (16 bytes
// each), exchanges them in registers and writes 8 x 16 bytes, instead of one
// 2-byte LDS store per element.  A block owns 16 MT output channels, 32 input
// channels and the three taps of one row dy; X is staged once per dx with the
// pixels outside the image as zeros, so every fragment is an aligned 16-byte
// LDS read.  Each wave takes a quarter of the staged pixels and the whole tile
// (MT x 6 MFMAs from MT + 6 reads a step); the four waves' sums are added in
// order at the end.  The next 128 pixels' loads are in flight meanwhile.
struct WgradArgs {
    const uint16_t *X, *dY;
    float *out;  // dW, or the split's partial sums
    int P, H, W, C, N, chunk;
};

// 8 consecutive channels of one row at byte offset o; channels >= n (n <= 8) and
// rows at kOutside read as zero.  mode: 2 16-byte rows, 1 even row length, 0 any.
__device__ __forceinline__ uint4 load_channels(__amdgpu_buffer_rsrc_t r, unsigned o, int n, int mode) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    if (mode == 2) {
        const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, int(o), 0, 0));
        return make_uint4(v.x, v.y, v.z, v.w);
    }
    unsigned v[4] = {0, 0, 0, 0};
    if (o & 0x80000000u) return make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (mode == 1) {
            if (2 * i < n) v[i] = unsigned(__builtin_amdgcn_raw_buffer_load_b32(r, int(o) + 4 * i, 0, 0));
        } else {
            if (2 * i < n) v[i] = uint16_t(__builtin_amdgcn_raw_buffer_load_b16(r, int(o) + 4 * i, 0, 0));
            if (2 * i + 1 < n)
                v[i] |= unsigned(uint16_t(__builtin_amdgcn_raw_buffer_load_b16(r, int(o) + 4 * i + 2, 0, 0))) << 16;
        }
    }
    return make_uint4(v[0], v[1], v[2], v[3]);
}

constexpr int kWgradPx = 128;
constexpr int64_t WGRAD_BLOCKS = 3;  // blocks a CU: its LDS holds three (43.5 KB each)

template <int MT>
__global__ __launch_bounds__(256) void k_wgrad(WgradArgs a) {
    constexpr int CO = 16 * MT, PITCH = kWgradPx + 8, G = kWgradPx / 8;
    constexpr int kA = G * CO / 8, kB = 3 * G * 4, R = (kA + kB + 255) / 256;
    constexpr unsigned kOutside = 0x80000000u;
    constexpr int kStage = (CO + 96) * PITCH * 2, kSums = 4 * 6 * 256 * 4;
    __shared__ __align__(16) unsigned char smem[kStage > kSums ? kStage : kSums];
    uint16_t *const sA = reinterpret_cast<uint16_t *>(smem);  // [CO][PITCH]
    uint16_t *const sB = sA + CO * PITCH;                     // [3][32][PITCH]
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, col = lane & 15;
    // block: (co tile, c tile, dy) of blockIdx.x
    const int nc = (a.C + 31) / 32;
    int b = blockIdx.x;
    const int dy = b % 3 - 1;
    b /= 3;
    const int c0 = (b % nc) * 32, co0 = (b / nc) * CO;
    const int beg = blockIdx.y * a.chunk, end = min(a.P, beg + a.chunk);

    __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(a.X), 0, int(unsigned(a.P) * unsigned(a.C) * 2u), 0x00020000);
    __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(a.dY), 0, int(unsigned(a.P) * unsigned(a.N) * 2u), 0x00020000);
    const int mx = a.C % 8 == 0 ? 2 : (a.C % 2 == 0 ? 1 : 0), my = a.N % 8 == 0 ? 2 : (a.N % 2 == 0 ? 1 : 0);

    uint4 r[R][8];
    auto fetch = [&](int pb) {
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int it = t + q * 256;
            if (it < kA) {
                const int g = it / (CO / 8), ch = co0 + (it % (CO / 8)) * 8;
                const int p = pb + g * 8;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const bool in = p + j < end && ch < a.N;
                    const unsigned o = in ? (unsigned(p + j) * unsigned(a.N) + unsigned(ch)) * 2u : kOutside;
                    r[q][j] = load_channels(yr, o, a.N - ch, my);
                }
            } else if (it < kA + kB) {
                const int i = it - kA, dx = i / (G * 4) - 1, g = (i / 4) % G, ch = c0 + (i % 4) * 8;
                const int p = pb + g * 8;
                int x = p % a.W, y = (p / a.W) % a.H;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const bool in = p + j < end && ch < a.C && unsigned(x + dx) < unsigned(a.W) &&
                                    unsigned(y + dy) < unsigned(a.H);
                    const unsigned o =
                        in ? (unsigned(p + j + dy * a.W + dx) * unsigned(a.C) + unsigned(ch)) * 2u : kOutside;
                    r[q][j] = load_channels(xr, o, a.C - ch, mx);
                    if (++x == a.W) {
                        x = 0;
                        if (++y == a.H) y = 0;
                    }
                }
            }
        }
    };
    auto stage = [&]() {
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int it = t + q * 256;
            if (it >= kA + kB) continue;
            uint16_t *d;  // row of the item's first channel
            if (it < kA) d = sA + (it % (CO / 8)) * 8 * PITCH + (it / (CO / 8)) * 8;
            else d = sB + ((it - kA) / (G * 4) * 32 + ((it - kA) % 4) * 8) * PITCH + ((it - kA) / 4 % G) * 8;
            const unsigned *v = reinterpret_cast<const unsigned *>(r[q]);
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                // channel c of pixels 2i and 2i + 1
                unsigned o[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    o[i] = __builtin_amdgcn_perm(v[(2 * i + 1) * 4 + c / 2], v[2 * i * 4 + c / 2],
                                                 c % 2 ? 0x07060302u : 0x05040100u);
                *reinterpret_cast<uint4 *>(d + c * PITCH) = make_uint4(o[0], o[1], o[2], o[3]);
            }
        }
    };

    floatx4 acc[MT][6];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < 6; ++n) acc[m][n] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int k = w * 32 + (lane >> 4) * 8;  // the lane's pixels of a stage
    fetch(beg);
    for (int pb = beg; pb < end; pb += kWgradPx) {
        stage();
        __syncthreads();
        if (pb + kWgradPx < end) fetch(pb + kWgradPx);
        bf16x8 x[6];
#pragma unroll
        for (int n = 0; n < 6; ++n)  // n = 2 dx + c tile
            x[n] = *reinterpret_cast<const bf16x8 *>(sB + (n * 16 + col) * PITCH + k);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const bf16x8 y = *reinterpret_cast<const bf16x8 *>(sA + (m * 16 + col) * PITCH + k);
#pragma unroll
            for (int n = 0; n < 6; ++n)
                acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y, x[n], acc[m][n], 0, 0, 0);
        }
        __syncthreads();
    }

    float *const sums = reinterpret_cast<float *>(smem);  // [wave][n][16 x 16]
    float *const out = a.out + int64_t(blockIdx.y) * a.N * 9 * a.C;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
        for (int n = 0; n < 6; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                sums[(w * 6 + n) * 256 + ((lane >> 4) * 4 + i) * 16 + col] = acc[m][n][i];
        __syncthreads();
#pragma unroll
        for (int n = 0; n < 6; ++n) {
            const float v = ((sums[n * 256 + t] + sums[(6 + n) * 256 + t]) + sums[(12 + n) * 256 + t]) +
                            sums[(18 + n) * 256 + t];
            const int co = co0 + m * 16 + (t >> 4), c = c0 + (n & 1) * 16 + (t & 15);
            if (co < a.N && c < a.C)
                out[(int64_t(co) * 9 + (dy + 1) * 3 + n / 2) * a.C + c] = v;
        }
        __syncthreads();
    }
}

// out = sum of k_wgrad's partials (splits x n values).  32 values a block and 8
// threads a value, each adding every eighth partial in order: there are few
// values and hundreds of partials, and one thread a value waits for one load
// after another (28 us a layer; 64 partials took 13).
__global__ __launch_bounds__(256) void k_wgrad_reduce(const float *__restrict__ work, int n, int splits,
                                                      float *__restrict__ out) {
    __shared__ float part[8][32];
    const int e = threadIdx.x & 31, g = threadIdx.x >> 5;
    const int i = blockIdx.x * 32 + e;
    float v = 0.0f;
    if (i < n) {
#pragma unroll 4
        for (int z = g; z < splits; z += 8) v += work[int64_t(z) * n + i];
    }
    part[g][e] = v;
    __syncthreads();
    if (g || i >= n) return;
#pragma unroll
    for (int q = 1; q < 8; ++q) v += part[q][e];
    out[i] = v;
}

// im2col for 3x3 same convolution: x [B][H][W][C] BF16 -> cols [B*H*W][9*C].
// Tap (dy, dx) = (blockIdx.y / 3, blockIdx.y % 3); each thread moves VEC
// consecutive channels of one pixel (VEC = 8: one 16-byte load and store,
// used when C % 8 == 0).  Indices are 32-bit: the caller checks B*H*W*C < 2^31.
template <int VEC>
__global__ __launch_bounds__(256) void k_im2col(const uint16_t *__restrict__ x, int H, int W, int C,
                                                uint16_t *__restrict__ cols, int items) {
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= items) return;  // items = B*H*W*C/VEC
    const int cv = C / VEC;
    const int c = (idx % cv) * VEC;
    const int p = idx / cv;
    const int xw = p % W, r = p / W;
    const int yh = r % H, b = r / H;
    const int tap = blockIdx.y;
    const int yy = yh + tap / 3 - 1, xx = xw + tap % 3 - 1;
    const bool inside = yy >= 0 && yy < H && xx >= 0 && xx < W;
    const int64_t src = ((int64_t(b) * H + yy) * W + xx) * C + c;
    const int64_t dst = (int64_t(p) * 9 + tap) * C + c;
    if constexpr (VEC == 8) {
        uint4 v = make_uint4(0, 0, 0, 0);
        if (inside) v = *reinterpret_cast<const uint4 *>(x + src);
        *reinterpret_cast<uint4 *>(cols + dst) = v;
    } else {
        cols[dst] = inside ? x[src] : uint16_t(0);
    }
}

// col2im (gather): dx[b][y][x][c] (+)= sum over taps of dcols[pixel(y - dy + 1, x - dx + 1)][tap*C + c].
__global__ __launch_bounds__(256) void k_col2im(const float *__restrict__ dcols, int B, int H, int W,
                                                int C, float *__restrict__ dx, int accumulate) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    const int64_t total = int64_t(B) * H * W * C;
    if (idx >= total) return;
    const int c = int(idx % C);
    int64_t r = idx / C;
    const int xw = int(r % W);
    const int64_t r2 = r / W;
    const int yh = int(r2 % H);
    const int b = int(r2 / H);
    float s = 0.0f;
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
        const int py = yh - (tap / 3 - 1), px = xw - (tap % 3 - 1);  // output pixel that read (yh, xw) at this tap
        if (py < 0 || py >= H || px < 0 || px >= W) continue;
        s += dcols[(((int64_t(b) * H + py) * W + px) * 9 + tap) * C + c];
    }
    dx[idx] = accumulate ? dx[idx] + s : s;
}

// dy *= (y > 0); writes a BF16 copy of the masked gradient.
__global__ __launch_bounds__(256) void k_relu_backward(const float *__restrict__ y, float *__restrict__ dy,
                                                       uint16_t *__restrict__ dyb, int64_t n) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const float g = y[i] > 0.0f ? dy[i] : 0.0f;
    dy[i] = g;
    if (dyb) dyb[i] = f2bf(g);
}

// db[n] = sum_m dy[m][n] in two fixed-order passes.  Pass 1: block b sums
// rows [b*rows, (b+1)*rows) of columns [c0, c0 + cw), cw = min(N - c0, 256);
// thread t owns column c0 + t % cw and rows t / cw, + 256 / cw, ... (coalesced
// across a row), the threads of one column are then added in LDS in order.
constexpr int kBiasBlocks = 1024;

__global__ __launch_bounds__(256) void k_bias_grad_partial(const float *__restrict__ dy, int64_t M,
                                                           int N, int c0, int64_t rows,
                                                           double *__restrict__ partial) {
    __shared__ double red[256];
    const int cw = min(N - c0, 256), t = threadIdx.x;
    const int lanes = 256 / cw;  // threads per column
    const int col = t % cw, r0 = t / cw;
    double s = 0.0;
    if (r0 < lanes) {
        const int64_t beg = int64_t(blockIdx.x) * rows, end = min(M, beg + rows);
        for (int64_t m = beg + r0; m < end; m += lanes) s += double(dy[m * N + c0 + col]);
    }
    red[t] = s;
    __syncthreads();
    if (t < cw) {
        double v = 0.0;
        for (int j = 0; j < lanes; ++j) v += red[j * cw + t];
        partial[int64_t(blockIdx.x) * N + c0 + t] = v;
    }
}

// Pass 1 of a layer's backward epilogue: g = dy where y > 0 (y null: everywhere),
// its BF16 copy, and the partial column sums of g in the same pass.  Four
// columns a thread (N % 4 == 0): 16-byte loads, and enough of them in flight.
// The masked FP32 gradient itself has no reader and is not written.
__global__ __launch_bounds__(256) void k_grad_epilogue(const float *__restrict__ y, const float *__restrict__ dy,
                                                       int64_t M, int N, int c0, int64_t rows,
                                                       uint16_t *__restrict__ dyb,
                                                       double *__restrict__ partial) {
    __shared__ double red[4][256];
    const int cw = min(N - c0, 256) / 4, t = threadIdx.x;  // column groups
    const int lanes = 256 / cw, cg = t % cw, r0 = t / cw;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (r0 < lanes) {
        const int64_t beg = int64_t(blockIdx.x) * rows, end = min(M, beg + rows);
#pragma unroll 4
        for (int64_t m = beg + r0; m < end; m += lanes) {
            const int64_t o = m * N + c0 + cg * 4;
            float4 g = *reinterpret_cast<const float4 *>(dy + o);
            if (y) {
                const float4 v = *reinterpret_cast<const float4 *>(y + o);
                g.x = v.x > 0.0f ? g.x : 0.0f;
                g.y = v.y > 0.0f ? g.y : 0.0f;
                g.z = v.z > 0.0f ? g.z : 0.0f;
                g.w = v.w > 0.0f ? g.w : 0.0f;
            }
            *reinterpret_cast<ushort4 *>(dyb + o) = make_ushort4(f2bf(g.x), f2bf(g.y), f2bf(g.z), f2bf(g.w));
            s[0] += double(g.x);
            s[1] += double(g.y);
            s[2] += double(g.z);
            s[3] += double(g.w);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) red[i][t] = s[i];
    __syncthreads();
    if (t < cw) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            double v = 0.0;
            for (int j = 0; j < lanes; ++j) v += red[i][j * cw + t];
            partial[int64_t(blockIdx.x) * N + c0 + t * 4 + i] = v;
        }
    }
}

// Pass 2: block n adds the nblocks partials of column n, one per thread at a
// time, in a fixed-shape tree, so all of them are loaded at once instead of
// one after another by a single thread.
__global__ __launch_bounds__(256) void k_bias_grad_final(const double *__restrict__ partial, int N,
                                                         int nblocks, float *__restrict__ db) {
    const int n = blockIdx.x, t = threadIdx.x;
    double v = 0.0;
    for (int b = t; b < nblocks; b += 256) v += partial[int64_t(b) * N + n];
    const double tot = block_sum(v);
    if (t == 0) db[n] = float(tot);
}

// Weights W[cout][tap][cin] -> Wt[cin][tap][cout] (BF16): the weights of the data
// gradient as a convolution of dY, k contiguous.
__global__ __launch_bounds__(256) void k_transpose_weights(const uint16_t *__restrict__ w, int cin,
                                                           int cout, uint16_t *__restrict__ wt) {
    const int i = blockIdx.x * 256 + threadIdx.x;  // over cin, tap, cout
    if (i >= 9 * cout * cin) return;
    const int co = i % cout, r = i / cout;
    const int tap = r % 9, c = r / 9;
    wt[i] = w[(int64_t(co) * 9 + tap) * cin + c];
}

// Weights W[cout][tap][cin] -> Wf[tap][cout][cin] (BF16): the B operand of the
// data gradient as a general GEMM (the form that the others are tested against),
// dX[p][c] = sum over (tap, co) of dY[p - tap][co] Wf[tap][co][c].
__global__ __launch_bounds__(256) void k_flip_weights(const uint16_t *__restrict__ w, int cin,
                                                      int cout, uint16_t *__restrict__ wf) {
    const int i = blockIdx.x * 256 + threadIdx.x;  // over tap, cout, cin
    if (i >= 9 * cout * cin) return;
    const int c = i % cin, r = i / cin;
    const int co = r % cout, tap = r / cout;
    wf[i] = w[(int64_t(co) * 9 + tap) * cin + c];
}

// V channels of one pixel: 4 (16-byte words) where the channel counts, offsets
// and pointers allow it, else 1.  These kernels move memory and little else; with
// one channel a thread they were bound by their index arithmetic (the network's
// three upsamplings at batch 16: 27.5 us on average against 12.4; channel
// copies 14.9 against 10.4, the pool's backward 15.3 against 7.4).
template <int V>
struct Vec {
    float v[V];
    __device__ __forceinline__ static Vec load(const float *p) {
        Vec r;
        if constexpr (V == 4) {
            const float4 q = *reinterpret_cast<const float4 *>(p);
            r.v[0] = q.x, r.v[1] = q.y, r.v[2] = q.z, r.v[3] = q.w;
        } else {
            r.v[0] = *p;
        }
        return r;
    }
    __device__ __forceinline__ void store(float *p) const {
        if constexpr (V == 4) *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
        else *p = v[0];
    }
    __device__ __forceinline__ void store_bf16(uint16_t *p) const {
        if constexpr (V == 4)
            *reinterpret_cast<ushort4 *>(p) = make_ushort4(f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3]));
        else *p = f2bf(v[0]);
    }
};

// Pixel and channel of item idx of a [B][H][W][C] array taken V channels at a time.
struct Pixel {
    int c, x, y, b;
    int64_t p;
    __device__ __forceinline__ Pixel(int64_t idx, int cv, int V, int H, int W) {
        c = int(idx % cv) * V;
        p = idx / cv;
        x = int(p % W);
        const int64_t r = p / W;
        y = int(r % H);
        b = int(r / H);
    }
};

// 2x2 average pool (NHWC): y [B][H/2][W/2][C].
template <int V>
__global__ __launch_bounds__(256) void k_avgpool2(const float *__restrict__ x, int B, int H, int W, int C,
                                                  float *__restrict__ y, uint16_t *__restrict__ yb) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= int64_t(B) * (H / 2) * (W / 2) * (C / V)) return;
    const Pixel o(idx, C / V, V, H / 2, W / 2);
    const float *p = x + ((int64_t(o.b) * H + 2 * o.y) * W + 2 * o.x) * C + o.c;
    const Vec<V> q0 = Vec<V>::load(p), q1 = Vec<V>::load(p + C);
    const Vec<V> q2 = Vec<V>::load(p + int64_t(W) * C), q3 = Vec<V>::load(p + int64_t(W) * C + C);
    Vec<V> r;
#pragma unroll
    for (int i = 0; i < V; ++i) r.v[i] = 0.25f * ((q0.v[i] + q1.v[i]) + (q2.v[i] + q3.v[i]));
    if (y) r.store(y + idx * V);
    if (yb) r.store_bf16(yb + idx * V);
}

template <int V>
__global__ __launch_bounds__(256) void k_avgpool2_backward(const float *__restrict__ dy, int B, int H,
                                                           int W, int C, float *__restrict__ dx,
                                                           int accumulate) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= int64_t(B) * H * W * (C / V)) return;
    const Pixel o(idx, C / V, V, H, W);
    Vec<V> g = Vec<V>::load(dy + ((int64_t(o.b) * (H / 2) + o.y / 2) * (W / 2) + o.x / 2) * C + o.c);
#pragma unroll
    for (int i = 0; i < V; ++i) g.v[i] = 0.25f * g.v[i];
    if (accumulate) {
        const Vec<V> q = Vec<V>::load(dx + idx * V);
#pragma unroll
        for (int i = 0; i < V; ++i) g.v[i] = q.v[i] + g.v[i];
    }
    g.store(dx + idx * V);
}

// Nearest 2x upsample of x [B][H][W][C] into channels [coff, coff + C) of
// y [B][2H][2W][Ct].
template <int V>
__global__ __launch_bounds__(256) void k_upsample2(const float *__restrict__ x, int B, int H, int W,
                                                   int C, float *__restrict__ y,
                                                   uint16_t *__restrict__ yb, int Ct, int coff) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= int64_t(B) * 4 * H * W * (C / V)) return;
    const Pixel o(idx, C / V, V, 2 * H, 2 * W);
    const Vec<V> v = Vec<V>::load(x + ((int64_t(o.b) * H + o.y / 2) * W + o.x / 2) * C + o.c);
    v.store(y + o.p * Ct + coff + o.c);
    if (yb) v.store_bf16(yb + o.p * Ct + coff + o.c);
}

template <int V>
__global__ __launch_bounds__(256) void k_upsample2_backward(const float *__restrict__ dy, int B, int H,
                                                            int W, int C, int Ct, int coff,
                                                            float *__restrict__ dx) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= int64_t(B) * H * W * (C / V)) return;
    const Pixel o(idx, C / V, V, H, W);
    Vec<V> s;
#pragma unroll
    for (int i = 0; i < V; ++i) s.v[i] = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int yo = 2 * o.y + q / 2, xo = 2 * o.x + q % 2;
        const Vec<V> g = Vec<V>::load(dy + ((int64_t(o.b) * (2 * H) + yo) * (2 * W) + xo) * Ct + coff + o.c);
#pragma unroll
        for (int i = 0; i < V; ++i) s.v[i] += g.v[i];
    }
    s.store(dx + idx * V);
}

// The decoder's input in BF16: nearest 2x upsample of h [B][H][W][Ch], then skip
// [B][2H][2W][Cs], V channels (16 bytes, or one) a thread.
template <int V>
__global__ __launch_bounds__(256) void k_concat_up(const uint16_t *__restrict__ h, const uint16_t *__restrict__ skip,
                                                   int64_t items, int H, int W, int Ch, int Cs,
                                                   uint16_t *__restrict__ out) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= items) return;
    const Pixel o(idx, (Ch + Cs) / V, V, 2 * H, 2 * W);
    const uint16_t *src = o.c < Ch ? h + ((int64_t(o.b) * H + o.y / 2) * W + o.x / 2) * Ch + o.c
                                   : skip + o.p * Cs + (o.c - Ch);
    if constexpr (V == 8) *reinterpret_cast<uint4 *>(out + idx * 8) = *reinterpret_cast<const uint4 *>(src);
    else out[idx] = *src;
}

// Channel-slice copy: dst[p][doff + c] (+)= src[p][soff + c] for c < C.
template <int V>
__global__ __launch_bounds__(256) void k_copy_channels(const float *__restrict__ src, int Cs, int soff,
                                                       float *__restrict__ dst, uint16_t *__restrict__ dstb,
                                                       int Cd, int doff, int C, int64_t P, int accumulate) {
    const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
    const int cv = C / V;
    if (idx >= P * cv) return;
    const int c = int(idx % cv) * V;
    const int64_t p = idx / cv, o = p * Cd + doff + c;
    Vec<V> v = Vec<V>::load(src + p * Cs + soff + c);
    if (accumulate) {
        const Vec<V> q = Vec<V>::load(dst + o);
#pragma unroll
        for (int i = 0; i < V; ++i) v.v[i] += q.v[i];
    }
    v.store(dst + o);
    if (dstb) v.store_bf16(dstb + o);
}

// Mean squared error over n values: loss partials and dy = 2 (y - t) / n.
__global__ __launch_bounds__(kBlock) void k_mse(const float *__restrict__ y, const float *__restrict__ t,
                                                int64_t n, float *__restrict__ dy,
                                                double *__restrict__ partial) {
    double s = 0.0;
    const int64_t stride = int64_t(gridDim.x) * kBlock;
    for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride) {
        const float d = y[i] - t[i];
        s += double(d) * double(d);
        dy[i] = 2.0f * d / float(n);
    }
    const double tot = block_sum(s);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot / double(n);
}

// Large-scale error term: e_bar = mean of (y - t) over each f x f block of
// cells (per image and channel); loss partials of weight * mean(e_bar^2) and
// dy += weight * 2 e_bar / (n_blocks f^2) on every cell of the block.  One
// thread per block: each cell is written by exactly one thread.
__global__ __launch_bounds__(kBlock) void k_mse_pooled(const float *__restrict__ y,
                                                       const float *__restrict__ t, int B, int H,
                                                       int W, int C, int f, float weight,
                                                       float *__restrict__ dy,
                                                       double *__restrict__ partial) {
    const int Hb = H / f, Wb = W / f;
    const int64_t nb = int64_t(B) * Hb * Wb * C;
    const double inv = 1.0 / (double(f) * f);
    double s = 0.0;
    const int64_t stride = int64_t(gridDim.x) * kBlock;
    for (int64_t q = int64_t(blockIdx.x) * kBlock + threadIdx.x; q < nb; q += stride) {
        const int c = int(q % C);
        int64_t r = q / C;
        const int xb = int(r % Wb);
        r /= Wb;
        const int yb = int(r % Hb);
        const int b = int(r / Hb);
        const int64_t base = ((int64_t(b) * H + int64_t(yb) * f) * W + int64_t(xb) * f) * C + c;
        double e = 0.0;
        for (int i = 0; i < f; ++i)
            for (int j = 0; j < f; ++j) {
                const int64_t o = base + (int64_t(i) * W + j) * C;
                e += double(y[o]) - double(t[o]);
            }
        e *= inv;
        s += e * e;
        const float g = float(weight * 2.0 * e * inv / double(nb));
        for (int i = 0; i < f; ++i)
            for (int j = 0; j < f; ++j) dy[base + (int64_t(i) * W + j) * C] += g;
    }
    const double tot = block_sum(s);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot * double(weight) / double(nb);
}

// Adam on FP32 master weights, BF16 copy for the GEMMs.
__global__ __launch_bounds__(256) void k_adam(float *__restrict__ p, const float *__restrict__ g,
                                              float *__restrict__ m, float *__restrict__ v,
                                              uint16_t *__restrict__ pb, int64_t n, float lr, float b1,
                                              float b2, float eps, float c1, float c2) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p[i] = pi;
    if (pb) pb[i] = f2bf(pi);
}

// Exponential moving average of the parameters: ema = decay * ema + (1 - decay) * p.
__global__ __launch_bounds__(256) void k_ema(float *__restrict__ ema, const float *__restrict__ p,
                                             int64_t n, float decay) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) ema[i] = decay * ema[i] + (1.0f - decay) * p[i];
}

__global__ __launch_bounds__(256) void k_to_bf16(const float *__restrict__ x, uint16_t *__restrict__ y,
                                                 int64_t n) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

// ---------------------------------------------------------------------------
// Warm start: the surrogate's normalized fields q [m][m][3] =
// ((rho - 1) / U^2, ux / U, uy / U), averages over the cells of an m x m grid
// covering the cavity -> populations f (FP64, reference layout 9 x nx x ny) on
// nx x ny nodes.  Node (k, l) sits at cell coordinate (px, py) =
// ((k + 1/2) m / nx - 1/2, (l + 1/2) m / ny - 1/2); the walls lie on the faces
// px = -1/2, px = m - 1/2, py = -1/2 and the lid on py = m - 1/2.
// Reconstruction of the node values:
//   * default: bilinear between cell centres, clamped beyond the outermost;
//   * WALLS: bilinear, with ghost cells mirrored across each wall beyond the
//     outermost centres: velocity ghosts 2 u_wall - u_mirror (u_wall = 0 on the
//     walls, (1, 0) on the lid, in units of U), density ghosts equal to the
//     mirror cell, so profiles run into the wall values;
//   * CUBIC (with the same ghosts, any depth): the cell averages are first
//     turned into point values at the centres, u_c = q - c * lap(q) (5-point
//     Laplacian; an r x r node average of a smooth field is its centre value
//     plus c * lap with c = (r^2 - 1) / (24 r^2)), then interpolated with
//     separable Catmull-Rom cubics (exact for quadratics);
// then f = f_eq(rho, u) in the opt1 order; with NEQ, plus the first-order
// non-equilibrium part of the BGK post-collision state,
// (1 - omega) * (-3 w_i rho / omega) Q_i : S, with the strain rate S from
// central differences of the reconstructed velocity (one-sided at the walls).
constexpr int kWarmNeq = 1, kWarmWalls = 2, kWarmCubic = 4;

// q at cell (i, j); cells outside [0, m) are ghosts mirrored across the wall
// faces (requires i, j in [-m, 2m)).
__device__ __forceinline__ double cell(const float *__restrict__ q, int m, int ch, int i, int j) {
    const int ii = i < 0 ? -1 - i : (i >= m ? 2 * m - 1 - i : i);
    const int jj = j < 0 ? -1 - j : (j >= m ? 2 * m - 1 - j : j);
    double v = q[(int64_t(ii) * m + jj) * 3 + ch];
    if (ch == 0) return v;
    if (j != jj) v = ((j >= m && ch == 1) ? 2.0 : 0.0) - v;  // bottom wall / lid
    if (i != ii) v = -v;                                   // left / right wall
    return v;
}

__device__ __forceinline__ double bilerp(const float *__restrict__ q, int m, int ch, double px,
                                         double py, bool walls) {
    int i0, j0, i1, j1;
    if (walls) {
        px = fmin(fmax(px, -1.0), double(m));
        py = fmin(fmax(py, -1.0), double(m));
        i0 = min(int(floor(px)), m - 1);
        j0 = min(int(floor(py)), m - 1);
        i1 = i0 + 1;
        j1 = j0 + 1;
    } else {
        px = fmin(fmax(px, 0.0), double(m - 1));
        py = fmin(fmax(py, 0.0), double(m - 1));
        i0 = m < 2 ? 0 : min(int(px), m - 2);
        j0 = m < 2 ? 0 : min(int(py), m - 2);
        i1 = min(i0 + 1, m - 1);
        j1 = min(j0 + 1, m - 1);
    }
    const double tx = px - i0, ty = py - j0;
    const double a = cell(q, m, ch, i0, j0), b = cell(q, m, ch, i1, j0);
    const double c = cell(q, m, ch, i0, j1), d = cell(q, m, ch, i1, j1);
    return (1 - tx) * ((1 - ty) * a + ty * c) + tx * ((1 - ty) * b + ty * d);
}

__device__ __forceinline__ void catmull_rom(double t, double w[4]) {
    const double t2 = t * t, t3 = t2 * t;
    w[0] = 0.5 * (-t3 + 2.0 * t2 - t);
    w[1] = 0.5 * (3.0 * t3 - 5.0 * t2 + 2.0);
    w[2] = 0.5 * (-3.0 * t3 + 4.0 * t2 + t);
    w[3] = 0.5 * (t3 - t2);
}

// Point value at the centre of cell (i, j), i, j in [-2, m + 1].
__device__ __forceinline__ double point(const float *__restrict__ q, int m, int ch, int i, int j,
                                        double c) {
    const double v = cell(q, m, ch, i, j);
    const double lap = (cell(q, m, ch, i + 1, j) + cell(q, m, ch, i - 1, j)) +
                       (cell(q, m, ch, i, j + 1) + cell(q, m, ch, i, j - 1)) - 4.0 * v;
    return v - c * lap;
}

__device__ __forceinline__ double cubic(const float *__restrict__ q, int m, int ch, double px,
                                       double py, double c) {
    px = fmin(fmax(px, -0.5), double(m) - 0.5);
    py = fmin(fmax(py, -0.5), double(m) - 0.5);
    const int i0 = min(int(floor(px)), m - 1), j0 = min(int(floor(py)), m - 1);
    double wx[4], wy[4];
    catmull_rom(px - i0, wx);
    catmull_rom(py - j0, wy);
    double s = 0.0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        double r = 0.0;
#pragma unroll
        for (int b = 0; b < 4; ++b) r += wy[b] * point(q, m, ch, i0 - 1 + a, j0 - 1 + b, c);
        s += wx[a] * r;
    }
    return s;
}

struct Recon {
    int mode;  // 0 clamped bilinear, 1 wall-ghost bilinear, 2 cubic
    double c;  // deconvolution coefficient (cubic)
};

__device__ __forceinline__ double reconstruct(const float *q, int m, int ch, double px, double py,
                                              Recon r) {
    return r.mode == 2 ? cubic(q, m, ch, px, py, r.c) : bilerp(q, m, ch, px, py, r.mode == 1);
}

__device__ __forceinline__ void sample(const float *q, int m, int nx, int ny, int k, int l, double U,
                                       Recon rc, double &rho, double &ux, double &uy) {
    const double px = (k + 0.5) * m / nx - 0.5, py = (l + 0.5) * m / ny - 0.5;
    rho = 1.0 + U * U * reconstruct(q, m, 0, px, py, rc);
    ux = U * reconstruct(q, m, 1, px, py, rc);
    uy = U * reconstruct(q, m, 2, px, py, rc);
}

__global__ __launch_bounds__(kBlock) void k_warm_init(const float *__restrict__ q, int m, int nx, int ny,
                                                      double U, double omega, int neq, Recon rc,
                                                      double *__restrict__ f) {
    const int64_t j = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    const int64_t P = int64_t(nx) * ny;
    if (j >= P) return;
    const int k = int(j / ny), l = int(j - int64_t(k) * ny);
    double rho, ux, uy;
    sample(q, m, nx, ny, k, l, U, rc, rho, ux, uy);
    double feq[9];
    equilibrium_opt1(rho, ux, uy, feq);
    if (neq) {
        const int km = max(k - 1, 0), kp = min(k + 1, nx - 1), lm = max(l - 1, 0), lp = min(l + 1, ny - 1);
        double r_, uxm, uym, uxp, uyp, uxl, uyl, uxu, uyu;
        sample(q, m, nx, ny, km, l, U, rc, r_, uxm, uym);
        sample(q, m, nx, ny, kp, l, U, rc, r_, uxp, uyp);
        sample(q, m, nx, ny, k, lm, U, rc, r_, uxl, uyl);
        sample(q, m, nx, ny, k, lp, U, rc, r_, uxu, uyu);
        const double hx = double(max(kp - km, 1)), hy = double(max(lp - lm, 1));
        const double dxux = (uxp - uxm) / hx, dxuy = (uyp - uym) / hx;
        const double dyux = (uxu - uxl) / hy, dyuy = (uyu - uyl) / hy;
        const double sxx = dxux, syy = dyuy, sxy = 0.5 * (dyux + dxuy);
        const double fac = (1.0 - omega) * (-3.0 * rho / omega);
        const double w[9] = {4.0 / 9, 1.0 / 9, 1.0 / 9, 1.0 / 9, 1.0 / 9, 1.0 / 36, 1.0 / 36, 1.0 / 36, 1.0 / 36};
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            const double cx_ = cx(i), cy_ = cy(i);
            const double qs = (cx_ * cx_ - 1.0 / 3) * sxx + 2.0 * cx_ * cy_ * sxy + (cy_ * cy_ - 1.0 / 3) * syy;
            feq[i] += fac * w[i] * qs;
        }
    }
#pragma unroll
    for (int i = 0; i < 9; ++i) f[i * P + j] = feq[i];
}

inline unsigned blocks_for(int64_t n, int per = 256) { return unsigned((n + per - 1) / per); }

}  // namespace nn
}  // namespace lbm

using namespace lbm;
using namespace lbm::nn;

extern "C" {

}  // extern "C"

// Tile-load form for an operand X(row, k) = X[row*s_row + k*s_k].
static int load_mode(const void *X, int64_t s_row, int64_t s_k) {
    const bool aligned = reinterpret_cast<uintptr_t>(X) % 16 == 0;
    if (aligned && s_k == 1 && s_row % 8 == 0) return LOAD_K;
    if (aligned && s_row == 1 && s_k % 8 == 0) return LOAD_ROW;
    return LOAD_SCALAR;
}

// Launch the GEMM (and the ordered split-K reduction when splits > 1).
static int run_gemm(const GemmArgs &g, int splits, hipStream_t s) {
    dim3 grid((g.N + TN - 1) / TN, (g.M + TM - 1) / TM, splits);
    hipLaunchKernelGGL(k_gemm, grid, dim3(256), 0, s, g);
    if (splits > 1)
        hipLaunchKernelGGL(k_gemm_reduce, dim3(blocks_for(int64_t(g.M) * g.N)), dim3(256), 0, s, g,
                           splits);
    return launch_status();
}

// Whether all counts are multiples of 4 and all pointers 16-byte aligned (8 for
// the BF16 ones): Vec<4>.
static bool by_four(std::initializer_list<int> counts, std::initializer_list<const void *> f32, const void *bf16) {
    for (int c : counts)
        if (c % 4) return false;
    for (const void *q : f32)
        if (reinterpret_cast<uintptr_t>(q) % 16) return false;
    return reinterpret_cast<uintptr_t>(bf16) % 8 == 0;
}

// k_conv3 where it applies: C a multiple of the 32 channels of a step, 16-byte
// aligned operands and (vector stores) outputs, operands below 2^31 bytes.
static bool conv_direct(const ConvArgs &a) {
    auto misaligned = [](const void *q) { return reinterpret_cast<uintptr_t>(q) % 16 != 0; };
    if (a.C % 32 || misaligned(a.X) || misaligned(a.Wt) || misaligned(a.y) || misaligned(a.yb)) return false;
    return int64_t(a.P) * a.C * 2 < (int64_t(1) << 31) && int64_t(a.N) * 9 * a.C * 2 < (int64_t(1) << 31);
}

// Output channels of a k_wgrad block: 64 where they divide evenly, else 32 (the
// staged X is shared by half as many, but none are computed for nothing).
static int wgrad_co(int cout) { return cout % 64 == 0 ? 64 : 32; }

// k_wgrad where its loads apply: offsets below 2^31 bytes, rows that are a multiple
// of 16 bytes on a 16-byte base, others on a 4-byte one.
static bool wgrad_direct(const void *x, const void *dy, int64_t P, int cin, int cout) {
    auto ok = [&](const void *q, int n) {
        return reinterpret_cast<uintptr_t>(q) % (n % 8 == 0 ? 16 : 4) == 0 && P * n * 2 < (int64_t(1) << 31);
    };
    return ok(x, cin) && ok(dy, cout);
}

static int run_conv(const ConvArgs &a, hipStream_t s) {
    // The largest tile that still gives every SIMD two waves: operands loaded per
    // MFMA fall with the tile, but a wave's 9 C / 32 steps are a serial chain.
    // 16 x 32 x 32, 256 -> 128: 4 x 2 tiles 54 us, 4 x 4 (one wave a SIMD) 73; batch 1,
    // 128 -> 128: 1 x 1 10.6 us, 2 x 2 19.8.
    const int64_t simds = 4 * int64_t(device_cus());
    auto waves = [&](int mt, int nt) {
        return int64_t((a.P + 16 * mt - 1) / (16 * mt)) * ((a.N + 16 * nt - 1) / (16 * nt));
    };
    auto launch = [&](auto kernel, int mt, int nt) {
        const dim3 grid(unsigned((a.P + 64 * mt - 1) / (64 * mt)), unsigned((a.N + 16 * nt - 1) / (16 * nt)));
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, a);
    };
    if (a.N > 32 && waves(4, 4) >= 2 * simds) launch(k_conv3<4, 4, 3>, 4, 4);
    else if (a.N > 16 && waves(4, 2) >= 2 * simds) launch(k_conv3<4, 2, 3>, 4, 2);
    else if (a.N > 16 && waves(2, 2) >= 2 * simds) launch(k_conv3<2, 2, 3>, 2, 2);
    else launch(k_conv3<1, 1, 9>, 1, 1);
    return launch_status();
}

// LDS of k_conv3p at 32 mt pixels a block, and the most a block may take: two
// share a CU.
static int64_t conv_lds(const ConvArgs &a, int mt) {
    return (int64_t(32) * mt + 2 * int64_t(a.W) + 3) * (2 * a.C + 16);
}
constexpr int64_t kConvLds = 80 * 1024;

// Elements of the packed weights of K summed and N output channels; 0 where the
// packed kernels do not apply (their offsets end at 2^31 bytes).
static int64_t packed_elements(int K, int N) {
    const int64_t n = K % 32 ? 0 : (int64_t(N) + 15) / 16 * 16 * 9 * K;
    return n < (int64_t(1) << 30) ? n : 0;
}

// The block of k_conv3p for a layer, 32 MT pixels x 32 NT channels as 10 MT + NT; 0
// where k_conv3 runs it.  us of layers (batch x side^2), and of k_conv3:
//   41, 128 x 32, where 64 channels would leave half of the last block's waves
//     without any (32 at most, or 65 to 96), from 3 blocks per two CUs.  32 -> 32 at
//     4 x 112^2 9.0 (22: 9.4, k_conv3 10.8), 3 x 128^2 9.1 (8.7, 9.8), 16 x 128^2
//     25.7 (30.0, 25.0); 96 -> 32 at 4 x 112^2 12.7 (22.0, 26.8), 8 x 128^2 32.9
//     (53.8, 31.7), 16 x 128^2 61.9 (102.6, 58.8); 96 -> 96 at 2 x 96^2 13.0 (17.4,
//     25.8), 16 x 128^2 161 (211, 134);
//   22, 64 x 64, while every CU gets a block: 256 -> 128 at 16 x 32^2 19.6 (66.0; 11:
//     40.1), 128 -> 128 13.0 (35.7; 18.7), 64 -> 64 at 16 x 64^2 16.6 (31.4; 27.2),
//     16 x 128^2 66.9 (84.6; 41: 83.9);
//   11, 32 x 32, the weights of nine steps in flight, below (128 -> 128 at 64^2 8.5,
//     22: 9.8, k_conv3 18.4) and where the rows leave the LDS no room for more, up
//     to six blocks a CU: 128 -> 32 at 3 x 128^2, 6 blocks, 37.9 (50.0), but 64 -> 64
//     at 256^2, 16 blocks, 70.3 (32.6), 64 -> 32, 8 blocks, 37.7 (21.8).
static int conv_packed_tile(const ConvArgs &a) {
    if (!conv_direct(a) || conv_lds(a, 1) > kConvLds || !packed_elements(a.C, a.N)) return 0;
    const int64_t cus = device_cus();
    auto blocks = [&](int mt, int nt) {
        return int64_t((a.P + 32 * mt - 1) / (32 * mt)) * ((a.N + 32 * nt - 1) / (32 * nt));
    };
    const bool half = a.N <= 32 || (a.N > 64 && a.N <= 96);
    if (half && conv_lds(a, 4) <= kConvLds && 2 * blocks(4, 1) >= 3 * cus) return 41;
    if (conv_lds(a, 2) <= kConvLds && blocks(2, 2) >= cus) return 22;
    return blocks(1, 1) <= 6 * cus ? 11 : 0;
}

template <int MT, int NT, int D>
static int launch_conv_packed(const ConvArgs &a, hipStream_t s) {
    const dim3 grid(unsigned((a.P + 32 * MT - 1) / (32 * MT)), unsigned((a.N + 32 * NT - 1) / (32 * NT)));
    hipLaunchKernelGGL((k_conv3p<MT, NT, D>), grid, dim3(256), unsigned(conv_lds(a, MT)), s, a);
    return launch_status();
}

static int run_conv_packed(const ConvArgs &a, int tile, hipStream_t s) {
    switch (tile) {
    case 41: return launch_conv_packed<4, 1, 3>(a, s);
    case 22: return launch_conv_packed<2, 2, 3>(a, s);
    default: return launch_conv_packed<1, 1, 9>(a, s);
    }
}

extern "C" {

int lbm_nn_packed_fits(int B, int H, int W, int cin, int cout) {
    const int64_t P = int64_t(B) * H * W;
    if (B <= 0 || H <= 0 || W <= 0 || cin <= 0 || cout <= 0 || P * 9 * cin >= (int64_t(1) << 31) ||
        P * cout >= (int64_t(1) << 31))
        return 0;
    const ConvArgs a{nullptr, nullptr, nullptr, nullptr, nullptr, int(P), H, W, cin, cout, 1, 0, 0};
    return conv_packed_tile(a) != 0;
}

int64_t lbm_nn_packed_size(int cin, int cout) {
    if (cin <= 0 || cout <= 0) return LBM_E_SIZE;
    const int64_t f = packed_elements(cin, cout), t = packed_elements(cout, cin);  // either orientation
    return f > t ? f : t;
}

int lbm_nn_pack_weights(const void *w, const int64_t *from, const int *cin, const int *cout, int n,
                        int transposed, void *out, const int64_t *to, void *stream) {
    if (!w || !from || !cin || !cout || !out || !to) return LBM_E_NULL;
    if (n <= 0 || n > LBM_NN_MAX_LAYERS) return LBM_E_SIZE;
    if (reinterpret_cast<uintptr_t>(out) % 16) return LBM_E_ARG;
    PackTable q{};
    q.transposed = transposed;
    for (int i = 0; i < n; ++i) {
        if (cin[i] <= 0 || cout[i] <= 0) return LBM_E_SIZE;
        if (from[i] < 0 || to[i] < 0 || to[i] % 8) return LBM_E_ARG;
        const int K = transposed ? cout[i] : cin[i], N = transposed ? cin[i] : cout[i];
        if (!packed_elements(K, N)) continue;
        const int j = q.n++;
        q.from[j] = from[i], q.to[j] = to[i], q.cin[j] = cin[i], q.cout[j] = cout[i];
        q.first[j + 1] = q.first[j] + ((N + 15) / 16 * (9 * K / 32) * 64 + 255) / 256;
    }
    if (q.n == 0) return LBM_OK;
    hipLaunchKernelGGL(k_pack_weights, dim3(unsigned(q.first[q.n])), dim3(256), 0, as_stream(stream),
                       static_cast<const uint16_t *>(w), static_cast<uint16_t *>(out), q);
    return launch_status();
}

}  // extern "C"

// The U-Net's layers and the buffers of one forward pass.
namespace {
struct Unet {
    struct Layer {
        int cin, cout, level;
        int64_t w, wp;  // element offsets in the flat parameters, in the packed ones
    };
    Layer layer[LBM_NN_MAX_LAYERS];
    int n = 0, levels = 0;
    int64_t packed = 0, bytes = 0;
    int64_t xb, encf, enca[8], skip[8], pool[8], mida, midb, cat[8], deca[8], decb[8];  // byte offsets
};

int64_t take(Unet &u, int64_t bytes) {
    const int64_t at = u.bytes;
    u.bytes += (bytes + 255) / 256 * 256;
    return at;
}

bool plan_unet(Unet &u, int B, int H, int W, int in_ch, const int *widths, int levels, int mid, int out_ch) {
    if (B <= 0 || H <= 0 || W <= 0 || in_ch <= 0 || mid <= 0 || out_ch <= 0 || !widths || levels < 1 ||
        levels > 7 || 4 * levels + 3 > LBM_NN_MAX_LAYERS || H % (1 << levels) || W % (1 << levels))
        return false;
    for (int i = 0; i < levels; ++i)
        if (widths[i] <= 0) return false;
    u.levels = levels;
    int64_t flat = 0;
    auto add = [&](int cin, int cout, int level) {
        u.layer[u.n++] = Unet::Layer{cin, cout, level, flat, u.packed};
        flat += int64_t(9) * cin * cout + cout;
        u.packed += packed_elements(cin, cout);
    };
    int c = in_ch;
    for (int i = 0; i < levels; ++i) add(c, widths[i], i), add(widths[i], widths[i], i), c = widths[i];
    add(c, mid, levels), add(mid, mid, levels), c = mid;
    for (int i = levels - 1; i >= 0; --i) add(c + widths[i], widths[i], i), add(widths[i], widths[i], i), c = widths[i];
    add(c, out_ch, 0);
    const int64_t P = int64_t(B) * H * W;
    (void)take(u, u.packed * 2);  // at 0
    u.xb = take(u, P * in_ch * 2);
    int64_t encf = 0;
    for (int i = 0; i < levels; ++i) {
        const int64_t p = P >> (2 * i);
        encf = encf > p * widths[i] * 4 ? encf : p * widths[i] * 4;
        u.enca[i] = take(u, p * widths[i] * 2);
        u.skip[i] = take(u, p * widths[i] * 2);
        u.pool[i] = take(u, p / 4 * widths[i] * 2);
        u.cat[i] = take(u, p * ((i + 1 < levels ? widths[i + 1] : mid) + widths[i]) * 2);
        u.deca[i] = take(u, p * widths[i] * 2);
        u.decb[i] = take(u, p * widths[i] * 2);
    }
    u.encf = take(u, encf);
    u.mida = take(u, (P >> (2 * levels)) * mid * 2);
    u.midb = take(u, (P >> (2 * levels)) * mid * 2);
    return true;
}
}  // namespace

extern "C" {

int64_t lbm_nn_unet_workspace(int B, int H, int W, int in_ch, const int *widths, int levels, int mid, int out_ch) {
    Unet u;
    return plan_unet(u, B, H, W, in_ch, widths, levels, mid, out_ch) ? u.bytes : int64_t(LBM_E_SIZE);
}

int lbm_nn_unet_forward(const float *x, int B, int H, int W, int in_ch, const int *widths, int levels, int mid,
                        int out_ch, const float *p, const void *pb, void *work, float *out, void *stream) {
    if (!x || !p || !pb || !work || !out) return LBM_E_NULL;
    Unet u;
    if (!plan_unet(u, B, H, W, in_ch, widths, levels, mid, out_ch)) return LBM_E_SIZE;
    if (reinterpret_cast<uintptr_t>(work) % 16) return LBM_E_ARG;
    char *const base = static_cast<char *>(work);
    const uint16_t *const wb = static_cast<const uint16_t *>(pb);
    int64_t from[LBM_NN_MAX_LAYERS], to[LBM_NN_MAX_LAYERS];
    int cin[LBM_NN_MAX_LAYERS], cout[LBM_NN_MAX_LAYERS];
    for (int i = 0; i < u.n; ++i)
        from[i] = u.layer[i].w, to[i] = u.layer[i].wp, cin[i] = u.layer[i].cin, cout[i] = u.layer[i].cout;
    int rc = lbm_nn_pack_weights(pb, from, cin, cout, u.n, 0, base, to, stream);
    if (!rc) rc = lbm_nn_to_bf16(x, base + u.xb, int64_t(B) * H * W * in_ch, stream);
    int next = 0;
    auto conv = [&](int64_t src, float *y, void *yb, bool relu) {
        const Unet::Layer &l = u.layer[next++];
        if (rc) return;
        const uint16_t *wp = l.cin % 32 ? nullptr : reinterpret_cast<const uint16_t *>(base) + l.wp;
        rc = lbm_nn_conv3x3_packed(base + src, B, H >> l.level, W >> l.level, l.cin, wb + l.w, wp, l.cout,
                                   p + l.w + int64_t(9) * l.cin * l.cout, y, yb, relu, stream);
    };
    float *const f32 = reinterpret_cast<float *>(base + u.encf);
    int64_t h = u.xb;
    for (int i = 0; i < levels; ++i) {
        conv(h, nullptr, base + u.enca[i], true);
        conv(u.enca[i], f32, base + u.skip[i], true);  // the pool averages the FP32 values
        const int hh = H >> i, ww = W >> i, c = widths[i];
        if (rc) return rc;
        const int64_t n = int64_t(B) * (hh / 2) * (ww / 2) * c;
        uint16_t *const pooled = reinterpret_cast<uint16_t *>(base + u.pool[i]);
        if (by_four({c}, {f32}, pooled))
            hipLaunchKernelGGL(k_avgpool2<4>, dim3(blocks_for(n / 4)), dim3(256), 0, as_stream(stream), f32, B, hh,
                               ww, c, static_cast<float *>(nullptr), pooled);
        else
            hipLaunchKernelGGL(k_avgpool2<1>, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), f32, B, hh, ww,
                               c, static_cast<float *>(nullptr), pooled);
        h = u.pool[i];
    }
    conv(h, nullptr, base + u.mida, true);
    conv(u.mida, nullptr, base + u.midb, true);
    h = u.midb;
    for (int i = levels - 1; i >= 0; --i) {
        if (rc) return rc;
        const int ch = i + 1 < levels ? widths[i + 1] : mid, cs = widths[i];
        const int64_t n = int64_t(B) * (H >> i) * (W >> i) * (ch + cs);
        const uint16_t *hp = reinterpret_cast<const uint16_t *>(base + h);
        const uint16_t *sp = reinterpret_cast<const uint16_t *>(base + u.skip[i]);
        uint16_t *cp = reinterpret_cast<uint16_t *>(base + u.cat[i]);
        if (ch % 8 == 0 && cs % 8 == 0)
            hipLaunchKernelGGL(k_concat_up<8>, dim3(blocks_for(n / 8)), dim3(256), 0, as_stream(stream), hp, sp,
                               n / 8, H >> (i + 1), W >> (i + 1), ch, cs, cp);
        else
            hipLaunchKernelGGL(k_concat_up<1>, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), hp, sp, n,
                               H >> (i + 1), W >> (i + 1), ch, cs, cp);
        conv(u.cat[i], nullptr, base + u.deca[i], true);
        conv(u.deca[i], nullptr, base + u.decb[i], true);
        h = u.decb[i];
    }
    conv(h, out, nullptr, false);
    return rc ? rc : launch_status();
}

int lbm_nn_conv3x3_packed(const void *x, int B, int H, int W, int cin, const void *w, const void *wp, int cout,
                          const float *bias, float *y, void *yb, int relu, void *stream) {
    if (!x || !w || (!y && !yb)) return LBM_E_NULL;
    if (B <= 0 || H <= 0 || W <= 0 || cin <= 0 || cout <= 0) return LBM_E_SIZE;
    const int64_t P = int64_t(B) * H * W;
    if (wp && P * 9 * cin < (int64_t(1) << 31) && P * cout < (int64_t(1) << 31)) {
        const ConvArgs a{static_cast<const uint16_t *>(x), static_cast<const uint16_t *>(wp), y,
                         static_cast<uint16_t *>(yb), bias, int(P), H, W, cin, cout, 1, 0, relu};
        if (const int tile = conv_packed_tile(a)) return run_conv_packed(a, tile, as_stream(stream));
    }
    return lbm_nn_conv3x3(x, B, H, W, cin, w, cout, bias, y, yb, relu, stream);
}

int lbm_nn_conv3x3_dgrad_packed(const void *dy, const void *wp, int B, int H, int W, int cin, int cout,
                                float *dx, void *stream) {
    if (!dy || !wp || !dx) return LBM_E_NULL;
    if (B <= 0 || H <= 0 || W <= 0 || cin <= 0 || cout <= 0) return LBM_E_SIZE;
    const int64_t P = int64_t(B) * H * W;
    if (P * 9 * cout >= (int64_t(1) << 31) || P * cin >= (int64_t(1) << 31)) return LBM_E_SIZE;
    const ConvArgs a{static_cast<const uint16_t *>(dy), static_cast<const uint16_t *>(wp), dx, nullptr,
                     nullptr, int(P), H, W, cout, cin, -1, 0, 0};
    const int tile = conv_packed_tile(a);
    return tile ? run_conv_packed(a, tile, as_stream(stream)) : LBM_E_ARG;
}

int64_t lbm_nn_gemm_workspace(int M, int N, int ksplit) {
    return ksplit > 1 ? int64_t(ksplit) * M * N * int64_t(sizeof(float)) : 0;
}

int lbm_nn_gemm(const void *A, int64_t sam, int64_t sak, const void *B, int64_t sbk, int64_t sbn,
                float *C, void *Cb, int64_t ldc, const float *bias, int M, int N, int K,
                int accumulate, int relu, int ksplit, float *work, void *stream) {
    if (!A || !B || (!C && !Cb)) return LBM_E_NULL;
    if (M <= 0 || N <= 0 || K <= 0 || ksplit <= 0) return LBM_E_SIZE;
    if (accumulate && !C) return LBM_E_ARG;
    if (ksplit > 1 && !work) return LBM_E_WORKSPACE;
    int kchunk = (K + ksplit - 1) / ksplit;
    kchunk = (kchunk + TK - 1) / TK * TK;
    const int splits = (K + kchunk - 1) / kchunk;
    GemmArgs g{static_cast<const uint16_t *>(A), sam, sak, static_cast<const uint16_t *>(B), sbk, sbn,
               C, static_cast<uint16_t *>(Cb), ldc, bias, M, N, K, kchunk, accumulate, relu, work,
               load_mode(A, sam, sak), load_mode(B, sbn, sbk), Gather{1, 1, 1, 0},
               Gather{1, 1, 1, 0}};
    return run_gemm(g, splits, as_stream(stream));
}

int lbm_nn_conv3x3(const void *x, int B, int H, int W, int cin, const void *w, int cout,
                   const float *bias, float *y, void *yb, int relu, void *stream) {
    if (!x || !w || (!y && !yb)) return LBM_E_NULL;
    if (B <= 0 || H <= 0 || W <= 0 || cin <= 0 || cout <= 0) return LBM_E_SIZE;
    const int64_t P = int64_t(B) * H * W;
    if (P * 9 * cin >= (int64_t(1) << 31) || P * cout >= (int64_t(1) << 31)) return LBM_E_SIZE;
    if (cin % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16) return LBM_E_ARG;
    const ConvArgs a{static_cast<const uint16_t *>(x), static_cast<const uint16_t *>(w), y,
                     static_cast<uint16_t *>(yb), bias, int(P), H, W, cin, cout, 1, 0, relu};
    if (conv_direct(a)) return run_conv(a, as_stream(stream));
    const int K = 9 * cin;
    GemmArgs g{static_cast<const uint16_t *>(x), 0, 0, static_cast<const uint16_t *>(w), 1, K, y,
               static_cast<uint16_t *>(yb), cout, bias, int(P), cout, K, (K + TK - 1) / TK * TK, 0,
               relu, nullptr, LOAD_SCALAR, load_mode(w, K, 1), Gather{H, W, cin, 1},
               Gather{1, 1, 1, 0}};
    return run_gemm(g, 1, as_stream(stream));
}

int lbm_nn_conv3x3_wgrad_splits(int B, int H, int W, int cin, int cout) {
    if (B <= 0 || H <= 0 || W <= 0 || cin <= 0 || cout <= 0) return LBM_E_SIZE;
    const int64_t P = int64_t(B) * H * W, chunks = (P + kWgradPx - 1) / kWgradPx;
    const int64_t co = wgrad_co(cout);
    const int64_t tiles = 3 * ((cin + 31) / 32) * ((cout + co - 1) / co);
    int64_t splits = (WGRAD_BLOCKS * int64_t(device_cus()) + tiles - 1) / tiles;
    if (splits > (chunks + 3) / 4) splits = (chunks + 3) / 4;
    return int(splits < 1 ? 1 : splits);
}

int lbm_nn_conv3x3_wgrad(const void *x, const void *dy, int B, int H, int W, int cin, int cout,
                         float *dw, int ksplit, float *work, void *stream) {
    if (!x || !dy || !dw) return LBM_E_NULL;
    if (B <= 0 || H <= 0 || W <= 0 || cin <= 0 || cout <= 0 || ksplit <= 0) return LBM_E_SIZE;
    const int64_t P = int64_t(B) * H * W;
    if (P * 9 * cin >= (int64_t(1) << 31) || P * cout >= (int64_t(1) << 31)) return LBM_E_SIZE;
    if (cin % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16) return LBM_E_ARG;
    if (ksplit > 1 && !work) return LBM_E_WORKSPACE;
    const int K = int(P), N = 9 * cin;
    int kchunk = (K + ksplit - 1) / ksplit;
    const int unit = P >= 2 * kWgradPx && wgrad_direct(x, dy, P, cin, cout) ? kWgradPx : TK;
    kchunk = (kchunk + unit - 1) / unit * unit;
    const int splits = (K + kchunk - 1) / kchunk;
    if (unit == kWgradPx) {
        WgradArgs a{static_cast<const uint16_t *>(x), static_cast<const uint16_t *>(dy),
                    splits > 1 ? work : dw, K, H, W, cin, cout, kchunk};
        const int co = wgrad_co(cout);
        const dim3 grid(unsigned(3 * ((cin + 31) / 32) * ((cout + co - 1) / co)), unsigned(splits));
        hipStream_t s = as_stream(stream);
        if (co == 64) hipLaunchKernelGGL(k_wgrad<4>, grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL(k_wgrad<2>, grid, dim3(256), 0, s, a);
        if (splits > 1) {
            hipLaunchKernelGGL(k_wgrad_reduce, dim3(blocks_for(int64_t(cout) * N, 32)), dim3(256), 0, s, work,
                               cout * N, splits, dw);
        }
        return launch_status();
    }
    GemmArgs g{static_cast<const uint16_t *>(dy), 1, cout, static_cast<const uint16_t *>(x), 0, 0,
               dw, nullptr, N, nullptr, cout, N, K, kchunk, 0, 0, work, load_mode(dy, 1, cout),
               LOAD_SCALAR, Gather{1, 1, 1, 0}, Gather{H, W, cin, 1}};
    return run_gemm(g, splits, as_stream(stream));
}

int lbm_nn_conv3x3_flip_weights(const void *w, int cin, int cout, void *wf, void *stream) {
    if (!w || !wf) return LBM_E_NULL;
    if (cin <= 0 || cout <= 0) return LBM_E_SIZE;
    hipLaunchKernelGGL(k_flip_weights, dim3(blocks_for(int64_t(9) * cout * cin)), dim3(256), 0,
                       as_stream(stream), static_cast<const uint16_t *>(w), cin, cout,
                       static_cast<uint16_t *>(wf));
    return launch_status();
}

int lbm_nn_conv3x3_dgrad(const void *dy, const void *wf, int B, int H, int W, int cin, int cout,
                         float *dx, int accumulate, void *stream) {
    if (!dy || !wf || !dx) return LBM_E_NULL;
    if (B <= 0 || H <= 0 || W <= 0 || cin <= 0 || cout <= 0) return LBM_E_SIZE;
    const int64_t P = int64_t(B) * H * W;
    if (P * 9 * cout >= (int64_t(1) << 31) || P * cin >= (int64_t(1) << 31)) return LBM_E_SIZE;
    if (cout % 8 == 0 && reinterpret_cast<uintptr_t>(dy) % 16) return LBM_E_ARG;
    const int K = 9 * cout;
    GemmArgs g{static_cast<const uint16_t *>(dy), 0, 0, static_cast<const uint16_t *>(wf), cin, 1,
               dx, nullptr, cin, nullptr, int(P), cin, K, (K + TK - 1) / TK * TK, accumulate, 0,
               nullptr, LOAD_SCALAR, load_mode(wf, 1, cin), Gather{H, W, cout, -1},
               Gather{1, 1, 1, 0}};
    return run_gemm(g, 1, as_stream(stream));
}

int lbm_nn_conv3x3_transpose_weights(const void *w, int cin, int cout, void *wt, void *stream) {
    if (!w || !wt) return LBM_E_NULL;
    if (cin <= 0 || cout <= 0) return LBM_E_SIZE;
    hipLaunchKernelGGL(k_transpose_weights, dim3(blocks_for(int64_t(9) * cout * cin)), dim3(256), 0,
                       as_stream(stream), static_cast<const uint16_t *>(w), cin, cout,
                       static_cast<uint16_t *>(wt));
    return launch_status();
}

int lbm_nn_conv3x3_dgrad_t(const void *dy, const void *wt, int B, int H, int W, int cin, int cout,
                           float *dx, int accumulate, void *stream) {
    if (!dy || !wt || !dx) return LBM_E_NULL;
    if (B <= 0 || H <= 0 || W <= 0 || cin <= 0 || cout <= 0) return LBM_E_SIZE;
    const int64_t P = int64_t(B) * H * W;
    if (P * 9 * cout >= (int64_t(1) << 31) || P * cin >= (int64_t(1) << 31)) return LBM_E_SIZE;
    if (cout % 8 == 0 && reinterpret_cast<uintptr_t>(dy) % 16) return LBM_E_ARG;
    const ConvArgs a{static_cast<const uint16_t *>(dy), static_cast<const uint16_t *>(wt), dx, nullptr,
                     nullptr, int(P), H, W, cout, cin, -1, accumulate, 0};
    if (conv_direct(a)) return run_conv(a, as_stream(stream));
    const int K = 9 * cout;
    GemmArgs g{static_cast<const uint16_t *>(dy), 0, 0, static_cast<const uint16_t *>(wt), 1, K,
               dx, nullptr, cin, nullptr, int(P), cin, K, (K + TK - 1) / TK * TK, accumulate, 0,
               nullptr, LOAD_SCALAR, load_mode(wt, K, 1), Gather{H, W, cout, -1},
               Gather{1, 1, 1, 0}};
    return run_gemm(g, 1, as_stream(stream));
}

int lbm_nn_im2col3x3(const void *x, int B, int H, int W, int C, void *cols, void *stream) {
    if (!x || !cols) return LBM_E_NULL;
    if (B <= 0 || H <= 0 || W <= 0 || C <= 0) return LBM_E_SIZE;
    const int64_t n = int64_t(B) * H * W * C;
    if (n >= (int64_t(1) << 31)) return LBM_E_SIZE;
    const bool vec = (C % 8 == 0) && (reinterpret_cast<uintptr_t>(x) % 16 == 0) &&
                     (reinterpret_cast<uintptr_t>(cols) % 16 == 0);
    const int items = int(vec ? n / 8 : n);
    dim3 grid(blocks_for(items), 9);
    hipStream_t s = as_stream(stream);
    if (vec)
        hipLaunchKernelGGL(k_im2col<8>, grid, dim3(256), 0, s, static_cast<const uint16_t *>(x), H, W, C,
                           static_cast<uint16_t *>(cols), items);
    else
        hipLaunchKernelGGL(k_im2col<1>, grid, dim3(256), 0, s, static_cast<const uint16_t *>(x), H, W, C,
                           static_cast<uint16_t *>(cols), items);
    return launch_status();
}

int lbm_nn_col2im3x3(const float *dcols, int B, int H, int W, int C, float *dx, int accumulate,
                     void *stream) {
    if (!dcols || !dx) return LBM_E_NULL;
    if (B <= 0 || H <= 0 || W <= 0 || C <= 0) return LBM_E_SIZE;
    hipLaunchKernelGGL(k_col2im, dim3(blocks_for(int64_t(B) * H * W * C)), dim3(256), 0,
                       as_stream(stream), dcols, B, H, W, C, dx, accumulate);
    return launch_status();
}

int lbm_nn_relu_backward(const float *y, float *dy, void *dy_bf16, int64_t n, void *stream) {
    if (!y || !dy) return LBM_E_NULL;
    if (n <= 0) return LBM_E_SIZE;
    hipLaunchKernelGGL(k_relu_backward, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), y, dy,
                       static_cast<uint16_t *>(dy_bf16), n);
    return launch_status();
}

int64_t lbm_nn_bias_grad_workspace(int N) { return int64_t(kBiasBlocks) * N * int64_t(sizeof(double)); }

int lbm_nn_bias_grad(const float *dy, int64_t M, int N, float *db, double *work, void *stream) {
    if (!dy || !db || !work) return LBM_E_NULL;
    if (M <= 0 || N <= 0) return LBM_E_SIZE;
    hipStream_t s = as_stream(stream);
    const int64_t rows = (M + kBiasBlocks - 1) / kBiasBlocks;
    const int nb = int((M + rows - 1) / rows);
    for (int c0 = 0; c0 < N; c0 += 256)
        hipLaunchKernelGGL(k_bias_grad_partial, dim3(nb), dim3(256), 0, s, dy, M, N, c0, rows, work);
    hipLaunchKernelGGL(k_bias_grad_final, dim3(N), dim3(256), 0, s, work, N, nb, db);
    return launch_status();
}

int lbm_nn_grad_epilogue(const float *y, float *dy, void *dy_bf16, int64_t M, int N, float *db,
                         double *work, void *stream) {
    if (!dy || !dy_bf16 || !db || !work) return LBM_E_NULL;
    if (M <= 0 || N <= 0) return LBM_E_SIZE;
    hipStream_t s = as_stream(stream);
    const bool vec = N % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(dy) % 16 == 0 && reinterpret_cast<uintptr_t>(dy_bf16) % 8 == 0;
    if (!vec) {
        const int rc = y ? lbm_nn_relu_backward(y, dy, dy_bf16, M * N, stream)
                         : lbm_nn_to_bf16(dy, dy_bf16, M * N, stream);
        return rc ? rc : lbm_nn_bias_grad(dy, M, N, db, work, stream);
    }
    const int64_t rows = (M + kBiasBlocks - 1) / kBiasBlocks;
    const int nb = int((M + rows - 1) / rows);
    for (int c0 = 0; c0 < N; c0 += 256)
        hipLaunchKernelGGL(k_grad_epilogue, dim3(nb), dim3(256), 0, s, y, dy, M, N, c0, rows,
                           static_cast<uint16_t *>(dy_bf16), work);
    hipLaunchKernelGGL(k_bias_grad_final, dim3(N), dim3(256), 0, s, work, N, nb, db);
    return launch_status();
}

int lbm_nn_avgpool2(const float *x, int B, int H, int W, int C, float *y, void *yb, void *stream) {
    if (!x || !y) return LBM_E_NULL;
    if (B <= 0 || H < 2 || W < 2 || C <= 0 || (H & 1) || (W & 1)) return LBM_E_SIZE;
    const int64_t n = int64_t(B) * (H / 2) * (W / 2) * C;
    if (by_four({C}, {x, y}, yb))
        hipLaunchKernelGGL(k_avgpool2<4>, dim3(blocks_for(n / 4)), dim3(256), 0, as_stream(stream), x, B, H, W,
                           C, y, static_cast<uint16_t *>(yb));
    else
        hipLaunchKernelGGL(k_avgpool2<1>, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), x, B, H, W, C,
                           y, static_cast<uint16_t *>(yb));
    return launch_status();
}

int lbm_nn_avgpool2_backward(const float *dy, int B, int H, int W, int C, float *dx, int accumulate,
                             void *stream) {
    if (!dy || !dx) return LBM_E_NULL;
    if (B <= 0 || H < 2 || W < 2 || C <= 0 || (H & 1) || (W & 1)) return LBM_E_SIZE;
    const int64_t n = int64_t(B) * H * W * C;
    if (by_four({C}, {dy, dx}, nullptr))
        hipLaunchKernelGGL(k_avgpool2_backward<4>, dim3(blocks_for(n / 4)), dim3(256), 0, as_stream(stream), dy,
                           B, H, W, C, dx, accumulate);
    else
        hipLaunchKernelGGL(k_avgpool2_backward<1>, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), dy, B,
                           H, W, C, dx, accumulate);
    return launch_status();
}

int lbm_nn_upsample2(const float *x, int B, int H, int W, int C, float *y, void *yb, int Ct, int coff,
                     void *stream) {
    if (!x || !y) return LBM_E_NULL;
    if (B <= 0 || H <= 0 || W <= 0 || C <= 0 || coff < 0 || coff + C > Ct) return LBM_E_SIZE;
    const int64_t n = int64_t(B) * 4 * H * W * C;
    if (by_four({C, Ct, coff}, {x, y}, yb))
        hipLaunchKernelGGL(k_upsample2<4>, dim3(blocks_for(n / 4)), dim3(256), 0, as_stream(stream), x, B, H, W,
                           C, y, static_cast<uint16_t *>(yb), Ct, coff);
    else
        hipLaunchKernelGGL(k_upsample2<1>, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), x, B, H, W, C,
                           y, static_cast<uint16_t *>(yb), Ct, coff);
    return launch_status();
}

int lbm_nn_upsample2_backward(const float *dy, int B, int H, int W, int C, int Ct, int coff,
                              float *dx, void *stream) {
    if (!dy || !dx) return LBM_E_NULL;
    if (B <= 0 || H <= 0 || W <= 0 || C <= 0 || coff < 0 || coff + C > Ct) return LBM_E_SIZE;
    const int64_t n = int64_t(B) * H * W * C;
    if (by_four({C, Ct, coff}, {dy, dx}, nullptr))
        hipLaunchKernelGGL(k_upsample2_backward<4>, dim3(blocks_for(n / 4)), dim3(256), 0, as_stream(stream),
                           dy, B, H, W, C, Ct, coff, dx);
    else
        hipLaunchKernelGGL(k_upsample2_backward<1>, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), dy, B,
                           H, W, C, Ct, coff, dx);
    return launch_status();
}

int lbm_nn_copy_channels(const float *src, int Cs, int soff, float *dst, void *dst_bf16, int Cd,
                         int doff, int C, int64_t P, int accumulate, void *stream) {
    if (!src || !dst) return LBM_E_NULL;
    if (C <= 0 || P <= 0 || soff < 0 || doff < 0 || soff + C > Cs || doff + C > Cd) return LBM_E_SIZE;
    if (by_four({C, Cs, soff, Cd, doff}, {src, dst}, dst_bf16))
        hipLaunchKernelGGL(k_copy_channels<4>, dim3(blocks_for(P * C / 4)), dim3(256), 0, as_stream(stream),
                           src, Cs, soff, dst, static_cast<uint16_t *>(dst_bf16), Cd, doff, C, P, accumulate);
    else
        hipLaunchKernelGGL(k_copy_channels<1>, dim3(blocks_for(P * C)), dim3(256), 0, as_stream(stream), src, Cs,
                           soff, dst, static_cast<uint16_t *>(dst_bf16), Cd, doff, C, P, accumulate);
    return launch_status();
}

int lbm_nn_mse(const float *y, const float *t, int64_t n, float *dy, double *work, double *loss,
               void *stream) {
    if (!y || !t || !dy || !work || !loss) return LBM_E_NULL;
    if (n <= 0) return LBM_E_SIZE;
    hipStream_t s = as_stream(stream);
    hipLaunchKernelGGL(k_mse, dim3(kReduceBlocks), dim3(kBlock), 0, s, y, t, n, dy, work);
    launch_sum_pass2(work, kReduceBlocks, 0.0, loss, s);
    return launch_status();
}

int lbm_nn_mse_pooled(const float *y, const float *t, int B, int H, int W, int C, int f,
                      float weight, float *dy, double *work, double *loss, void *stream) {
    if (!y || !t || !dy || !work || !loss) return LBM_E_NULL;
    if (B <= 0 || H <= 0 || W <= 0 || C <= 0 || f <= 0 || H % f || W % f) return LBM_E_SIZE;
    hipStream_t s = as_stream(stream);
    hipLaunchKernelGGL(k_mse_pooled, dim3(kReduceBlocks), dim3(kBlock), 0, s, y, t, B, H, W, C, f,
                       weight, dy, work);
    launch_sum_pass2(work, kReduceBlocks, 0.0, loss, s);
    return launch_status();
}

int lbm_nn_adam(float *p, const float *g, float *m, float *v, void *p_bf16, int64_t n, float lr,
                float b1, float b2, float eps, int step, void *stream) {
    if (!p || !g || !m || !v) return LBM_E_NULL;
    if (n <= 0 || step <= 0) return LBM_E_SIZE;
    const float c1 = 1.0f - powf(b1, float(step)), c2 = 1.0f - powf(b2, float(step));
    hipLaunchKernelGGL(k_adam, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), p, g, m, v,
                       static_cast<uint16_t *>(p_bf16), n, lr, b1, b2, eps, c1, c2);
    return launch_status();
}

int lbm_nn_ema(float *ema, const float *p, int64_t n, float decay, void *stream) {
    if (!ema || !p) return LBM_E_NULL;
    if (n <= 0) return LBM_E_SIZE;
    if (!(decay >= 0.0f && decay < 1.0f)) return LBM_E_ARG;
    hipLaunchKernelGGL(k_ema, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), ema, p, n, decay);
    return launch_status();
}

int lbm_nn_to_bf16(const float *x, void *y, int64_t n, void *stream) {
    if (!x || !y) return LBM_E_NULL;
    if (n <= 0) return LBM_E_SIZE;
    hipLaunchKernelGGL(k_to_bf16, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), x,
                       static_cast<uint16_t *>(y), n);
    return launch_status();
}

int lbm_warm_init_f64(const float *q, int m, int64_t nx, int64_t ny, double U, double omega,
                      int flags, int pool, double *f, void *stream) {
    if (!q || !f) return LBM_E_NULL;
    if (m <= 0 || !valid_grid(nx, ny)) return LBM_E_SIZE;
    if (!(U > 0.0) || !(omega > 0.0 && omega < 2.0) ||
        (flags & ~(kWarmNeq | kWarmWalls | kWarmCubic)) || pool < 1)
        return LBM_E_ARG;
    if ((flags & kWarmCubic) && m < 3) return LBM_E_SIZE;
    Recon rc{(flags & kWarmCubic) ? 2 : ((flags & kWarmWalls) ? 1 : 0),
             (double(pool) * pool - 1.0) / (24.0 * double(pool) * pool)};
    const int64_t P = nx * ny;
    hipLaunchKernelGGL(k_warm_init, dim3(blocks_for(P, kBlock)), dim3(kBlock), 0, as_stream(stream), q,
                       m, int(nx), int(ny), U, omega, int((flags & kWarmNeq) != 0), rc, f);
    return launch_status();
}

}  // extern "C"
