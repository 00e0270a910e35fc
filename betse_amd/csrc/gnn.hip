// gnn.hip -- kernels of the warm-start graph network (no counterpart in the
// reference): BF16 MFMA matrix products with FP32 accumulation, mean
// aggregation over the cell-adjacency graph and its adjoint, SiLU, masked MSE
// and Adam; for the usual widths whole passes with a kernel per layer. The C ABI is
// declared in include/betse_amd.h; where there are no layer kernels, the Python model in
// betse_amd/gnn.py composes the passes from the single calls.

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "betse_amd.h"

namespace {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef short v4s_lds __attribute__((ext_vector_type(4), may_alias));   // (LDS that holds either type)
typedef float v4f_lds __attribute__((ext_vector_type(4), may_alias));

constexpr int EB = 256;   // elementwise block

// float -> bfloat16 bits, round to nearest even (inputs are finite)
__device__ __forceinline__ short to_bf16(float x) {
    unsigned u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (short)(u >> 16);
}

// C tile (16 rows x 64 columns per block, one 16x16 tile per wavefront) of
// op(A) op(B) over k in [k_lo, k_hi), with v_mfma_f32_16x16x16bf16_1k.
// Lane l supplies A[r0 + l%16][k0 + 4*(l/16) + j] and B[k0 + 4*(l/16) + j][c0 + l%16],
// j = 0..3, and receives C[r0 + 4*(l/16) + q][c0 + l%16], q = 0..3.
__global__ void __launch_bounds__(256)
k_gemm_bf16(const float* __restrict__ A, long long sam, long long sak,
            const float* __restrict__ B, long long sbk, long long sbn,
            float* __restrict__ out, long long ldo, int m, int n, int kd, int kchunk) {
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int r0 = blockIdx.x * 16;
    const int c0 = blockIdx.y * 64 + wave * 16;
    const int k_lo = blockIdx.z * kchunk;
    const int k_hi = min(kd, k_lo + kchunk);
    if (c0 >= n) return;
    const int row = r0 + lane % 16, col = c0 + lane % 16, kq = 4 * (lane / 16);
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = k_lo; k0 < k_hi; k0 += 16) {
        v4s a, b;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = k0 + kq + j;
            const bool kin = (k < k_hi);
            a[j] = (kin && row < m) ? to_bf16(A[row * sam + k * sak]) : (short)0;
            b[j] = (kin && col < n) ? to_bf16(B[k * sbk + col * sbn]) : (short)0;
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
    float* o = out + (long long)blockIdx.z * m * (long long)ldo;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r = r0 + kq + q;
        if (r < m && col < n) o[r * ldo + col] = acc[q];
    }
}

// C (+)= sum of the split-K partials
__global__ void __launch_bounds__(EB)
k_sum_splits(const float* ws, int splits, float* C, long long ldc, int m, int n, int beta) {
    const long long e = (long long)blockIdx.x * EB + threadIdx.x;
    if (e >= (long long)m * n) return;
    const int r = (int)(e / n), c = (int)(e % n);
    float s = 0.f;
    for (int q = 0; q < splits; ++q) s += ws[(long long)q * m * n + (long long)r * n + c];
    C[r * ldc + c] = beta ? C[r * ldc + c] + s : s;
}

__device__ __forceinline__ float silu_f(float z) { return z / (1.f + expf(-z)); }

// Z += b; H = silu(Z) (+ Hres)
__global__ void __launch_bounds__(EB)
k_bias_silu(float* Z, const float* b, float* H, const float* Hres, int n, int f) {
    const long long e = (long long)blockIdx.x * EB + threadIdx.x;
    if (e >= (long long)n * f) return;
    const float z = Z[e] + b[e % f];
    Z[e] = z;
    const float s = silu_f(z);
    H[e] = Hres ? Hres[e] + s : s;
}

__global__ void __launch_bounds__(EB)
k_bias(float* Y, const float* b, int n, int f) {
    const long long e = (long long)blockIdx.x * EB + threadIdx.x;
    if (e < (long long)n * f) Y[e] += b[e % f];
}

// dZ = dH * silu'(Z)
__global__ void __launch_bounds__(EB)
k_silu_bwd(const float* dH, const float* Z, float* dZ, long long count) {
    const long long e = (long long)blockIdx.x * EB + threadIdx.x;
    if (e >= count) return;
    const float z = Z[e];
    const float s = 1.f / (1.f + expf(-z));
    dZ[e] = dH[e] * (s * (1.f + z * (1.f - s)));
}

// out[i] = mean_{j in N(i)} H[j]   (deg clamped to 1)
__global__ void __launch_bounds__(EB)
k_mean_agg(const float* H, long long ldh, const int32_t* ptr, const int32_t* idx, float* out, long long ldo,
           int n, int f) {
    const long long e = (long long)blockIdx.x * EB + threadIdx.x;
    if (e >= (long long)n * f) return;
    const int i = (int)(e / f), c = (int)(e % f);
    const int a = ptr[i], b = ptr[i + 1];
    float s = 0.f;
    for (int q = a; q < b; ++q) s += H[(long long)idx[q] * ldh + c];
    out[(long long)i * ldo + c] = s / (float)max(b - a, 1);
}

// adjoint on a symmetric graph: out[j] (+)= sum_{i in N(j)} G[i] / deg_i
__global__ void __launch_bounds__(EB)
k_mean_agg_T(const float* G, long long ldg, const int32_t* ptr, const int32_t* idx, float* out, long long ldo,
             int n, int f, int accumulate) {
    const long long e = (long long)blockIdx.x * EB + threadIdx.x;
    if (e >= (long long)n * f) return;
    const int j = (int)(e / f), c = (int)(e % f);
    float s = 0.f;
    for (int q = ptr[j]; q < ptr[j + 1]; ++q) {
        const int i = idx[q];
        s += G[(long long)i * ldg + c] / (float)max(ptr[i + 1] - ptr[i], 1);
    }
    float* o = out + (long long)j * ldo + c;
    *o = accumulate ? *o + s : s;
}

// column sums, two passes: per-block partials then a final reduction
__global__ void __launch_bounds__(EB)
k_colsum_part(const float* G, long long ldg, int n, int f, int rows_per_block, float* part) {
    const int c = threadIdx.x;
    if (c >= f) return;
    const int r0 = blockIdx.x * rows_per_block;
    const int r1 = min(n, r0 + rows_per_block);
    float s = 0.f;
    for (int r = r0; r < r1; ++r) s += G[(long long)r * ldg + c];
    part[(long long)blockIdx.x * f + c] = s;
}

__global__ void __launch_bounds__(EB)
k_colsum_final(const float* part, int parts, int f, float* out) {
    const int c = blockIdx.x * EB + threadIdx.x;
    if (c >= f) return;
    float s = 0.f;
    for (int q = 0; q < parts; ++q) s += part[(long long)q * f + c];
    out[c] = s;
}

// masked MSE: dY = 2 (Y - T) mask / count, per-block partial losses
__global__ void __launch_bounds__(EB)
k_mse(const float* Y, const float* T, const float* mask, long long count, float inv_n, float* dY, float* part) {
    __shared__ float red[EB];
    const long long e = (long long)blockIdx.x * EB + threadIdx.x;
    float l = 0.f;
    if (e < count) {
        const float d = (Y[e] - T[e]) * mask[e];
        dY[e] = 2.f * d * inv_n;
        l = d * d * inv_n;
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int s = EB / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// ---------------------------------------------------------------------------
// the whole network: one kernel per layer and direction
// ---------------------------------------------------------------------------
// One wavefront per 16 nodes computes the transposed product W^T h^T: a lane then
// holds four consecutive columns of one node both as an operand and as a result,
// so the neighbour sums, both products, bias, SiLU and residual stay in registers,
// every load and store is 16 bytes, and a layer's result is the next product's
// operand as it stands. Weights are rounded to BF16 once per block, in LDS in
// operand order. As products and elementwise calls a layer passed over its
// activations nine times forward and fourteen backward; now it reads them and the
// neighbours' once and writes what the backward pass reads. Every sum is in the
// order of those calls, so the results are the same bits. The eight XCDs take
// contiguous ranges of nodes: neighbours are near in the numbering, and each L2
// then holds the rows its own nodes gather.
// 160k nodes, 6 layers of 64: the forward pass 1,916 -> 140 us; a training step on 40k
// nodes 5,070 -> 366, on 800 nodes 1,264 -> 256. A layer's two passes over HBM and its
// vector instructions (SiLU, sums) take about as long as each other; 94-118 registers
// leave 16 wavefronts per CU.
constexpr int NB = 256, NW = NB / 64;        // threads and wavefronts per block
constexpr int NODES = 16;                    // nodes per wavefront
constexpr int64_t MAX_FLOATS = 1 << 30;      // of an activation: byte offsets of 32 bits
constexpr int NET_BLOCKS = 1024;             // blocks at most: four or more per CU

// 16 bytes of an array of fewer than 2^30 floats: 32-bit offsets, one register each
__device__ __forceinline__ v4f load4(const float* base, unsigned at) {
    return *reinterpret_cast<const v4f*>(reinterpret_cast<const char*>(base) + (size_t)(at * 4u));
}
__device__ __forceinline__ void store4(float* base, unsigned at, v4f v) {
    *reinterpret_cast<v4f*>(reinterpret_cast<char*>(base) + (size_t)(at * 4u)) = v;
}

// this wavefront's node tiles: [first, last) by stride
struct Tiles {
    int t, end, stride;
};
__device__ __forceinline__ Tiles my_tiles(int n) {
    const int T = (n + NODES - 1) / NODES, x = blockIdx.x % 8, per = gridDim.x / 8;
    const int lo = (int)((long long)T * x / 8), hi = (int)((long long)T * (x + 1) / 8);
    return {lo + (int)(blockIdx.x / 8) * NW + __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), hi, per * NW};
}

// to_bf16 by the conversion instruction (two values each)
__device__ __forceinline__ v4s bf16x4(v4f x) {
    typedef __bf16 v4b __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(v4s, __builtin_convertvector(x, v4b));
}

// s / d for an integer d < 2^26, r = 1.0 / d: a quotient of 24 bits by d is never so
// near the middle of two floats that the product's error of 2^-52 could cross it, so
// it rounds as the division does (three instructions instead of eleven). Below 2^-126,
// where floats have fewer bits, a quotient can lie in the middle and then be rounded up
// where the division rounds down, or down for up (the first such d is 98).
__device__ __forceinline__ float div_int(float s, double r) { return (float)((double)s * r); }

__device__ __forceinline__ v4f mfma16(v4s a, v4s b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// LDS operands of the product with op(W) (kd x nd): fragment [ks][ct][lane] holds
// op(W)[16 ks + 4 (lane/16) + j][16 ct + lane%16], zero outside
template <int K_TILES, int N_TILES>
__device__ __forceinline__ void stage_weights(v4s* s, const float* W, int sk, int sn, int kd, int nd) {
    constexpr int ITEMS = K_TILES * N_TILES * 64, PER = (ITEMS + NB - 1) / NB;
    // (a lane's four values in a row, whole and aligned: one load)
    const bool rows = sk == 1 && sn % 4 == 0 && kd == 16 * K_TILES && ITEMS % NB == 0 && ((size_t)W & 15) == 0;
    float x[PER][4];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int e = threadIdx.x + q * NB;
        const int lane = e % 64, ct = (e / 64) % N_TILES, ks = e / (64 * N_TILES);
        const int k = 16 * ks + 4 * (lane / 16), c = min(16 * ct + lane % 16, nd - 1);
        if (rows) {
            const v4f v = *reinterpret_cast<const v4f*>(W + k + (long long)c * sn);
#pragma unroll
            for (int j = 0; j < 4; ++j) x[q][j] = v[j];
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) x[q][j] = W[(long long)min(k + j, kd - 1) * sk + (long long)c * sn];
        }
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int e = threadIdx.x + q * NB;
        const int lane = e % 64, ct = (e / 64) % N_TILES, ks = e / (64 * N_TILES);
        const int k = 16 * ks + 4 * (lane / 16), c = 16 * ct + lane % 16;
        v4s v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (k + j < kd && c < nd) ? to_bf16(x[q][j]) : (short)0;
        if (ITEMS % NB == 0 || e < ITEMS) s[e] = v;
    }
}

// The lanes of a wavefront exchange values through LDS: what they stored before is what
// they load after. (It executes in order; this keeps the compiler from reordering.)
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// A wavefront's 16 nodes by H = 16 HB columns in two layouts: rows, where lane l
// holds columns 4 c4 .. 4 c4 + 3 (c4 = l % LR) of node it RI + l / LR in element it,
// consecutive lanes on consecutive addresses; and operands, where it holds columns
// 16 ks + 4 (l / 16) + 0..3 of node l % 16 in element ks. LDS turns one into the
// other (rows padded by one lane's piece: no bank conflicts). Loaded as operands, 16
// lanes on 16 rows, every lane is an access of its own to the vector memory's address
// unit: 41 us instead of 29 for 160k nodes.
template <int HB>
struct Tile {
    static constexpr int LR = 4 * HB, RI = 64 / LR, PITCH = LR + 1;
    static constexpr int LDS = NODES * PITCH;            // of v4f
    int g, c4, node, kq;
    v4f_lds* f;                                          // this wavefront's LDS
    v4s_lds* b;
    __device__ __forceinline__ explicit Tile(v4f* lds) {
        const int lane = threadIdx.x % 64;
        g = lane / LR;
        c4 = lane % LR;
        node = lane % 16;
        kq = lane / 16;
        f = reinterpret_cast<v4f_lds*>(lds) + threadIdx.x / 64 * LDS;
        b = reinterpret_cast<v4s_lds*>(f);
    }
    // rows to BF16 operands (half 0 or 1 of the LDS)
    __device__ __forceinline__ void operands(v4s (&o)[HB], const v4f (&x)[HB], int half) {
        v4s_lds* t = b + half * LDS;
        wave_sync();
#pragma unroll
        for (int it = 0; it < HB; ++it) t[(it * RI + g) * PITCH + c4] = bf16x4(x[it]);
        wave_sync();
#pragma unroll
        for (int ks = 0; ks < HB; ++ks) o[ks] = t[node * PITCH + 4 * ks + kq];
    }
    // results to rows
    __device__ __forceinline__ void rows(v4f (&x)[HB], const v4f (&acc)[HB]) {
        wave_sync();
#pragma unroll
        for (int ct = 0; ct < HB; ++ct) f[node * PITCH + 4 * ct + kq] = acc[ct];
        wave_sync();
#pragma unroll
        for (int it = 0; it < HB; ++it) x[it] = f[(it * RI + g) * PITCH + c4];
    }
};

// sums of the neighbours' rows, in list order: a neighbour of each of the lane's
// nodes at a time (two were as fast on few nodes and 3 % slower on many: registers).
// a, b: the nodes' ranges of idx.
template <int HB>
__device__ __forceinline__ void gather(v4f (&s)[HB], const float* h, const int32_t* idx, const int (&a)[HB],
                                       const int (&b)[HB], int c4) {
    int deg = 0;
#pragma unroll
    for (int it = 0; it < HB; ++it) {
        s[it] = v4f{0.f, 0.f, 0.f, 0.f};
        deg = max(deg, b[it] - a[it]);
    }
    if (deg <= 0) return;
    // (past a node's last neighbour the last is loaded again and not added)
    auto at = [&](int it, int q) { return idx[max(min(a[it] + q, b[it] - 1), 0)]; };
    int nb[HB];
#pragma unroll
    for (int it = 0; it < HB; ++it) nb[it] = at(it, 0);
    for (int q = 0; q < deg; ++q) {
        v4f x[HB];
#pragma unroll
        for (int it = 0; it < HB; ++it) x[it] = load4(h, (unsigned)nb[it] * (16 * HB) + 4 * c4);
#pragma unroll
        for (int it = 0; it < HB; ++it) nb[it] = at(it, q + 1);
#pragma unroll
        for (int it = 0; it < HB; ++it) {
            const bool in = a[it] + q < b[it];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float t = s[it][j] + x[it][j];
                s[it][j] = in ? t : s[it][j];
            }
        }
    }
}

// h0 = silu(X W_in + b_in); z0 (may be NULL) its argument
template <int HB>
__global__ void __launch_bounds__(NB)
k_net_in(const float* X, int f_in, const float* W, const float* bias, float* z, float* h, int n) {
    constexpr int H = 16 * HB;
    extern __shared__ v4s s_w[];
    __shared__ v4f s_t[NW * Tile<HB>::LDS];
    const int k_tiles = (f_in + 15) / 16;
    for (int ks = 0; ks < k_tiles; ++ks)
        stage_weights<1, HB>(s_w + ks * HB * 64, W + (long long)ks * 16 * H, H, 1, f_in - 16 * ks, H);
    __syncthreads();
    Tile<HB> L(s_t);
    const int lane = threadIdx.x % 64;
    v4f bv;
#pragma unroll
    for (int j = 0; j < 4; ++j) bv[j] = bias[4 * L.c4 + j];
    const Tiles T = my_tiles(n);
    for (int t = T.t; t < T.end; t += T.stride) {
        const int row = min(t * NODES + L.node, n - 1);
        v4f acc[HB], x[HB];
#pragma unroll
        for (int ct = 0; ct < HB; ++ct) acc[ct] = v4f{0.f, 0.f, 0.f, 0.f};
        for (int ks = 0; ks < k_tiles; ++ks) {
            v4f v;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = 16 * ks + 4 * L.kq + j;
                const float w = X[(long long)row * f_in + min(k, f_in - 1)];
                v[j] = (k < f_in) ? w : 0.f;
            }
            const v4s b = bf16x4(v);
#pragma unroll
            for (int ct = 0; ct < HB; ++ct) acc[ct] = mfma16(s_w[(ks * HB + ct) * 64 + lane], b, acc[ct]);
        }
        L.rows(x, acc);
#pragma unroll
        for (int it = 0; it < HB; ++it) {
            const int r = t * NODES + it * L.RI + L.g;
            if (r >= n) continue;
            const unsigned o = (unsigned)r * H + 4 * L.c4;
            const v4f zz = x[it] + bv;
            v4f s;
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] = silu_f(zz[j]);
            if (z) store4(z, o, zz);
            store4(h, o, s);
        }
    }
}

// hn = h + silu(z), z = h Wa + mean_nbr(h) Wb + b; agg, z and hn are stored where
// not NULL; with y, also y = hn W_out + b_out (f_out <= 16)
template <int HB>
__global__ void __launch_bounds__(NB, 4)
k_net_layer(const float* h, const int32_t* ptr, const int32_t* idx, const float* W, const float* bias, float* agg, float* z,
            float* hn, const float* Wout, const float* bout, float* y, int f_out, int n) {
    constexpr int H = 16 * HB;
    __shared__ v4s s_w[2 * HB * HB * 64];
    __shared__ v4s s_o[HB * 64];
    __shared__ v4f s_t[NW * Tile<HB>::LDS];
    stage_weights<2 * HB, HB>(s_w, W, H, 1, 2 * H, H);
    if (y) stage_weights<HB, 1>(s_o, Wout, f_out, 1, H, f_out);
    __syncthreads();
    Tile<HB> L(s_t);
    const int lane = threadIdx.x % 64;
    v4f bv;
#pragma unroll
    for (int j = 0; j < 4; ++j) bv[j] = bias[4 * L.c4 + j];
    const Tiles T = my_tiles(n);
    for (int t = T.t; t < T.end; t += T.stride) {
        const int r0 = t * NODES + L.g;
        int a[HB], b[HB];
        v4f own[HB], s[HB], acc1[HB], acc2[HB];
#pragma unroll
        for (int it = 0; it < HB; ++it) {
            const int row = min(r0 + it * L.RI, n - 1);
            a[it] = ptr[row];
            b[it] = ptr[row + 1];
            own[it] = load4(h, (unsigned)row * H + 4 * L.c4);
            acc1[it] = acc2[it] = v4f{0.f, 0.f, 0.f, 0.f};
        }
        gather<HB>(s, h, idx, a, b, L.c4);
#pragma unroll
        for (int it = 0; it < HB; ++it) {
            const double inv_deg = 1.0 / (double)max(b[it] - a[it], 1);
#pragma unroll
            for (int j = 0; j < 4; ++j) s[it][j] = div_int(s[it][j], inv_deg);
            const int r = r0 + it * L.RI;
            if (agg && r < n) store4(agg, (unsigned)r * H + 4 * L.c4, s[it]);
        }
        v4s x[HB], m[HB];
        L.operands(x, own, 0);
        L.operands(m, s, 1);
#pragma unroll
        for (int ks = 0; ks < HB; ++ks) {
            asm volatile("" ::: "memory");       // operands stay in LDS: hoisted they spill
#pragma unroll
            for (int ct = 0; ct < HB; ++ct) {
                acc1[ct] = mfma16(s_w[(ks * HB + ct) * 64 + lane], x[ks], acc1[ct]);
                acc2[ct] = mfma16(s_w[((HB + ks) * HB + ct) * 64 + lane], m[ks], acc2[ct]);
            }
        }
#pragma unroll
        for (int ct = 0; ct < HB; ++ct)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc1[ct][j] = acc1[ct][j] + (0.f + acc2[ct][j]);
        L.rows(s, acc1);
#pragma unroll
        for (int it = 0; it < HB; ++it) {
            const int r = r0 + it * L.RI;
            const unsigned e = (unsigned)r * H + 4 * L.c4;
            const v4f zz = s[it] + bv;
#pragma unroll
            for (int j = 0; j < 4; ++j) own[it][j] = own[it][j] + silu_f(zz[j]);
            if (z && r < n) store4(z, e, zz);
            if (hn && r < n) store4(hn, e, own[it]);
        }
        if (y) {
            v4f o = {0.f, 0.f, 0.f, 0.f};
            L.operands(x, own, 0);
#pragma unroll
            for (int ks = 0; ks < HB; ++ks) o = mfma16(s_o[ks * 64 + lane], x[ks], o);
            const int r = t * NODES + L.node;
            if (r < n)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (4 * L.kq + j < f_out) y[(long long)r * f_out + 4 * L.kq + j] = o[j] + bout[4 * L.kq + j];
        }
    }
}

// One layer backwards. The gradient of its output, g, is dY W_out^T at the top
// (dY not NULL) and otherwise dH plus what the neighbours' aggregates send back,
// the sum of their G = dagg / deg (divided where it is written, once per node, as
// the sum divided each). dz = g silu'(z). Below the layer (W not NULL):
// dH = g + dz Wa^T, in place, and G_out = (dz Wb^T) / deg.
template <int HB>
__global__ void __launch_bounds__(NB, 4)
k_net_layer_bwd(const float* dY, const float* Wout, int f_out, float* dH, const float* G, const int32_t* ptr,
                const int32_t* idx, const float* z, const float* W, float* dz, float* G_out, int n) {
    constexpr int H = 16 * HB;
    __shared__ v4s s_w[2 * HB * HB * 64];
    __shared__ v4s s_o[HB * 64];
    __shared__ v4f s_t[NW * Tile<HB>::LDS];
    if (W) {
        stage_weights<HB, HB>(s_w, W, 1, H, H, H);
        stage_weights<HB, HB>(s_w + HB * HB * 64, W + H * H, 1, H, H, H);
    }
    if (dY) stage_weights<1, HB>(s_o, Wout, 1, f_out, f_out, H);
    __syncthreads();
    Tile<HB> L(s_t);
    const int lane = threadIdx.x % 64;
    const Tiles T = my_tiles(n);
    for (int t = T.t; t < T.end; t += T.stride) {
        const int r0 = t * NODES + L.g;
        int a[HB], b[HB];
        v4f g[HB], zz[HB], acc1[HB], acc2[HB];
#pragma unroll
        for (int it = 0; it < HB; ++it) {
            const int row = min(r0 + it * L.RI, n - 1);
            a[it] = ptr[row];
            b[it] = ptr[row + 1];
            zz[it] = load4(z, (unsigned)row * H + 4 * L.c4);
            if (!dY) g[it] = load4(dH, (unsigned)row * H + 4 * L.c4);
            acc1[it] = acc2[it] = v4f{0.f, 0.f, 0.f, 0.f};
        }
        if (dY) {
            const int row = min(t * NODES + L.node, n - 1);
            v4f x;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float w = dY[(long long)row * f_out + min(4 * L.kq + j, f_out - 1)];
                x[j] = (4 * L.kq + j < f_out) ? w : 0.f;
            }
            const v4s xb = bf16x4(x);
            v4f o[HB];
#pragma unroll
            for (int ct = 0; ct < HB; ++ct) o[ct] = mfma16(s_o[ct * 64 + lane], xb, v4f{0.f, 0.f, 0.f, 0.f});
            L.rows(g, o);
        }
        if (G) {
            v4f s[HB];
            gather<HB>(s, G, idx, a, b, L.c4);
#pragma unroll
            for (int it = 0; it < HB; ++it) g[it] += s[it];
        }
#pragma unroll
        for (int it = 0; it < HB; ++it) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float s = 1.f / (1.f + expf(-zz[it][j]));
                zz[it][j] = g[it][j] * (s * (1.f + zz[it][j] * (1.f - s)));
            }
            const int r = r0 + it * L.RI;
            if (r < n) store4(dz, (unsigned)r * H + 4 * L.c4, zz[it]);
        }
        if (!W) continue;
        v4s x[HB];
        L.operands(x, zz, 0);
#pragma unroll
        for (int ks = 0; ks < HB; ++ks) {
            asm volatile("" ::: "memory");
#pragma unroll
            for (int ct = 0; ct < HB; ++ct) {
                acc1[ct] = mfma16(s_w[(ks * HB + ct) * 64 + lane], x[ks], acc1[ct]);
                acc2[ct] = mfma16(s_w[((HB + ks) * HB + ct) * 64 + lane], x[ks], acc2[ct]);
            }
        }
        L.rows(zz, acc1);
#pragma unroll
        for (int it = 0; it < HB; ++it) {
            const int r = r0 + it * L.RI;
#pragma unroll
            for (int j = 0; j < 4; ++j) g[it][j] = g[it][j] + (0.f + zz[it][j]);
            if (r < n) store4(dH, (unsigned)r * H + 4 * L.c4, g[it]);
        }
        L.rows(zz, acc2);
#pragma unroll
        for (int it = 0; it < HB; ++it) {
            const int r = r0 + it * L.RI;
            const double inv_deg = 1.0 / (double)max(b[it] - a[it], 1);
#pragma unroll
            for (int j = 0; j < 4; ++j) zz[it][j] = div_int(zz[it][j], inv_deg);
            if (r < n) store4(G_out, (unsigned)r * H + 4 * L.c4, zz[it]);
        }
    }
}

// ---------------------------------------------------------------------------
// weight and bias gradients of all layers, one launch
// ---------------------------------------------------------------------------
// C = A^T B over the n nodes, in `splits` chunks of nodes whose partials are added
// in order, and column sums of B in chunks of 256 nodes. A block multiplies 32
// columns of A with 64 of B over one chunk: a serial chain of up to 4,096 nodes,
// so what counts is the bytes in flight: 128 nodes are loaded (16 bytes a lane)
// while the 128 before are multiplied from LDS, where they lie transposed in BF16.
// All layers' products together fill the chip; one at a time a layer had 40 blocks.
// 40k nodes, 6 layers of 64: 63 us with 190 MB to read once (as calls 2,600). Tiles of
// 32 x 32 took 67, one chunk in flight 64, three 72.
constexpr int WM = 32, WN = 64;              // columns of A and of B per block
constexpr int WK = 128;                      // nodes staged at a time
constexpr int WCOLS = 112;                   // LDS columns per group of four nodes: 96, padded so that groups 16 lanes apart use other banks
constexpr int COL_ROWS = 256;                // nodes per column-sum partial
// block barrier for LDS only: __syncthreads waits for the loads in flight as well
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr int MAX_PROBS = 32;                // products (and column sums) per launch

struct WProb {
    const float* A; const float* B; float* out;   // out: the partials, or the gradient itself (one split)
    int m, n;                                     // columns (and row strides) of A and B
    int first;                                    // its first block, counted in m-blocks per split
};
struct WColsum {
    const float* B; float* part; int f;
};
struct WArgs {
    WProb p[MAX_PROBS]; WColsum c[MAX_PROBS];
    int n_probs, m_blocks;                        // m_blocks: of all products, for one split
    int n_sums, parts, sum_blocks;                // sum_blocks: blocks of one column sum
    int nodes, kchunk, splits;
};

__global__ void __launch_bounds__(NB, 2)
k_net_wgrad(WArgs a) {
    __shared__ __align__(16) v4s lds[2][WK / 4][WCOLS];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const int n_sum = a.n_sums * a.sum_blocks;
    if ((int)blockIdx.x < n_sum) {
        // column sums: a wavefront per partial, a lane per column
        const int q = blockIdx.x / a.sum_blocks, part = (blockIdx.x - q * a.sum_blocks) * NW + wave;
        if (part >= a.parts) return;
        const WColsum S = a.c[q];
        const int r0 = part * COL_ROWS, r1 = min(a.nodes, r0 + COL_ROWS);
        for (int c = lane; c < S.f; c += 64) {
            float s = 0.f;
            const float* g = S.B + (long long)r0 * S.f + c;
            int r = r0;
            for (; r + 32 <= r1; r += 32, g += 32 * S.f) {
                float x[32];
#pragma unroll
                for (int j = 0; j < 32; ++j) x[j] = g[j * S.f];
#pragma unroll
                for (int j = 0; j < 32; ++j) s += x[j];
            }
            for (; r < r1; ++r, g += S.f) s += *g;
            S.part[(long long)part * S.f + c] = s;
        }
        return;
    }
    // products: the blocks of one chunk of nodes follow each other on one XCD,
    // whose L2 then holds the rows they share
    const int total = a.m_blocks * a.splits, per = (total + 7) / 8;
    const int v0 = blockIdx.x - n_sum, v = (v0 % 8) * per + v0 / 8;
    if (v0 / 8 >= per || v >= total) return;
    const int split = v / a.m_blocks, mb = v - split * a.m_blocks;
    int q = 0;
    while (q + 1 < a.n_probs && a.p[q + 1].first <= mb) ++q;
    const WProb P = a.p[q];
    const int m_per = (P.m + WM - 1) / WM, local = mb - P.first;
    const int c0 = (local % m_per) * WM, n0 = (local / m_per) * WN;
    const int k_lo = split * a.kchunk, k_hi = min(a.nodes, k_lo + a.kchunk);
    const bool va = P.m % 4 == 0 && ((size_t)P.A & 15) == 0, vb = P.n % 4 == 0 && ((size_t)P.B & 15) == 0;
    // a thread's items of four nodes by four columns: two of B, one of A
    constexpr int AHEAD = 2;                      // chunks in flight
    v4f xb[AHEAD][2][4], xa[AHEAD][4];
    const int gb = tid / 16, cb = 4 * (tid % 16), ga = tid / 8, ca = 4 * (tid % 8);
    const bool fa = va && c0 + WM <= P.m, fb = vb && n0 + WN <= P.n;
    // four nodes' columns c..c+3 of M (ld columns): addresses kept inside, values
    // outside zero, so that the loads need no branch and stay in flight together
    auto rows = [&](v4f (&x)[4], const float* M, int ld, int k, int c, bool vec) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float* row = M + (long long)min(k + j, k_hi - 1) * ld;
            if (vec) {
                x[j] = *reinterpret_cast<const v4f*>(row + c);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) x[j][i] = row[min(c + i, ld - 1)];
            }
        }
    };
    auto load = [&](v4f (&b)[2][4], v4f (&a4)[4], int k0) {
        if (k0 >= k_hi) return;
        rows(b[0], P.B, P.n, k0 + 4 * gb, n0 + cb, fb);
        rows(b[1], P.B, P.n, k0 + 4 * gb + 64, n0 + cb, fb);
        rows(a4, P.A, P.m, k0 + 4 * ga, c0 + ca, fa);
    };
    v4f acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    auto step = [&](int buf, int s) {
        const v4s* f = &lds[buf][4 * s + lane / 16][lane % 16];
        const v4s b = f[WM + wave * 16];
        acc[0] = mfma16(f[0], b, acc[0]);
        acc[1] = mfma16(f[16], b, acc[1]);
    };
    auto put = [&](v4f (&x)[4], int buf, int k0, int g, int at, int c, int ld, bool vec) {
        if (!vec || k0 + WK > k_hi)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) x[j][i] = (k0 + 4 * g + j < k_hi && c + i < ld) ? x[j][i] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) lds[buf][g][at + i] = bf16x4(v4f{x[0][i], x[1][i], x[2][i], x[3][i]});
    };
#pragma unroll
    for (int d = 0; d < AHEAD; ++d) load(xb[d], xa[d], k_lo + d * WK);
    int buf = 0;
    for (int kk = k_lo; kk < k_hi; kk += AHEAD * WK) {
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) {
            const int k0 = kk + d * WK;
            if (k0 < k_hi) {
                // (the buffer's readers of two chunks ago passed the last barrier)
                put(xb[d][0], buf, k0, gb, WM + cb, n0 + cb, P.n, fb);
                put(xb[d][1], buf, k0, gb + 16, WM + cb, n0 + cb, P.n, fb);
                put(xa[d], buf, k0, ga, ca, c0 + ca, P.m, fa);
                load(xb[d], xa[d], k0 + AHEAD * WK);
                lds_barrier();
                const int steps = min(WK / 16, (k_hi - k0 + 15) / 16);
                if (n0 + wave * 16 < P.n) {
                    if (steps == WK / 16) {
#pragma unroll
                        for (int s = 0; s < WK / 16; ++s) step(buf, s);
                    } else {
                        for (int s = 0; s < steps; ++s) step(buf, s);
                    }
                }
                buf ^= 1;
            }
        }
    }
    float* out = P.out + (long long)split * P.m * P.n;
    const int col = n0 + wave * 16 + lane % 16;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = c0 + 16 * u + 4 * (lane / 16) + j;
            if (r < P.m && col < P.n) out[(long long)r * P.n + col] = acc[u][j];
        }
}

// the partials' sums, in order: an element per thread
struct FinalSeg {
    const float* part; float* out; int len, parts, first;   // first: its first block
};
struct FinalArgs {
    FinalSeg s[2 * MAX_PROBS]; int n_segs;
};
__global__ void __launch_bounds__(64)
k_net_sums(FinalArgs a) {
    int q = 0;
    while (q + 1 < a.n_segs && a.s[q + 1].first <= (int)blockIdx.x) ++q;
    const FinalSeg S = a.s[q];
    const int e = (blockIdx.x - S.first) * 64 + threadIdx.x;
    if (e >= S.len) return;
    float s = 0.f;
    int p = 0;
    auto add = [&](auto count) {                  // count partials, their loads in flight together
        constexpr int N = decltype(count)::value;
        for (; p + N <= S.parts; p += N) {
            float x[N];
#pragma unroll
            for (int j = 0; j < N; ++j) x[j] = S.part[(long long)(p + j) * S.len + e];
#pragma unroll
            for (int j = 0; j < N; ++j) s += x[j];
        }
    };
    add(std::integral_constant<int, 64>());
    add(std::integral_constant<int, 8>());
    add(std::integral_constant<int, 1>());
    S.out[e] = s;
}

// Adam on several tensors
constexpr int MAX_TENSORS = 48;
struct AdamArgs {
    float* p[MAX_TENSORS]; const float* g[MAX_TENSORS]; float* m[MAX_TENSORS]; float* v[MAX_TENSORS];
    long long count[MAX_TENSORS]; int first[MAX_TENSORS];   // first: the tensor's first block
    int n; float lr, b1, b2, eps, c1, c2;
};
__global__ void __launch_bounds__(EB)
k_adam(AdamArgs a) {
    int q = 0;
    while (q + 1 < a.n && a.first[q + 1] <= (int)blockIdx.x) ++q;
    const long long e = (long long)(blockIdx.x - a.first[q]) * EB + threadIdx.x;
    if (e >= a.count[q]) return;
    const float gg = a.g[q][e];
    const float mm = a.b1 * a.m[q][e] + (1.f - a.b1) * gg;
    const float vv = a.b2 * a.v[q][e] + (1.f - a.b2) * gg * gg;
    a.m[q][e] = mm;
    a.v[q][e] = vv;
    a.p[q][e] -= a.lr * (mm / a.c1) / (sqrtf(vv / a.c2) + a.eps);
}

inline unsigned blocks(long long n) { return (unsigned)((n + EB - 1) / EB); }

}  // namespace

// Scratch of bt_gnn_colsum_noalloc: the per-block partial sums live in this
// file-scope device array instead of a caller workspace. Each GPU the library
// runs on holds its own copy until the process ends; host code reaches it only
// through the device address hipGetSymbolAddress returns for the current
// device (the array's name on the host is not a device address).
static __device__ __align__(256) float scratch[BT_GNN_SCRATCH_FLOATS];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
float* g_scratch[MAX_DEVICES] = {};

// the device address of `scratch` on the current device, looked up once per device
int scratch_address(float** out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return BT_EHIP;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch[dev]) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return BT_EHIP;
        g_scratch[dev] = static_cast<float*>(ptr);
    }
    *out = g_scratch[dev];
    return BT_OK;
}

// rows per partial-sum block of the column sums: 256, doubled until the
// partials (one row of f per block) fit in ws_len floats
int colsum_rows_per_block(int n, int f, long long ws_len) {
    int rpb = 256;
    int parts = (n + rpb - 1) / rpb;
    while ((long long)parts * f > ws_len) {
        rpb *= 2;
        parts = (n + rpb - 1) / rpb;
    }
    return rpb;
}

// the networks whose layers have kernels of their own: an output row within one
// 16-column tile; operands in registers up to 64 columns; a row of X of at most 128
// (its weights in LDS); and products enough for one launch
bool layered(int f_in, int f_out, int hidden, int n_layers) {
    return (hidden == 16 || hidden == 32 || hidden == 64) && f_out >= 1 && f_out <= 16 && f_in >= 1 && f_in <= 128 &&
           n_layers >= 1 && 2 * n_layers + 2 <= MAX_PROBS;
}

// chunks of nodes of the weight-gradient products
int node_chunk(int n) {
    const int ksplit = (n > 4096) ? std::min(64, (n + 4095) / 4096) : 1;
    return ((n + ksplit - 1) / ksplit + 15) / 16 * 16;
}
int node_splits(int n) { return (n + node_chunk(n) - 1) / node_chunk(n); }

unsigned net_blocks(int n) {
    const int tiles = (n + NODES - 1) / NODES;
    return (unsigned)std::min(NET_BLOCKS, ((tiles + NW - 1) / NW + 7) / 8 * 8);
}

// params and grads: W_in, b_in, then W and b of each layer, then W_out, b_out.
// cache: h_0..h_L, z_0..z_L, agg_0..agg_{L-1} (keep), or two of h
template <int HB>
void net_forward(const float* const* params, int f_in, int f_out, int L, const float* X, const int32_t* ptr,
                 const int32_t* idx, int n, float* cache, bool keep, float* y, hipStream_t s) {
    constexpr int H = 16 * HB;
    const size_t row = (size_t)n * H;
    float* const hs = cache;
    float* const zs = cache + (L + 1) * row;
    float* const as = zs + (L + 1) * row;
    const dim3 grid(net_blocks(n));
    const size_t lds = (size_t)((f_in + 15) / 16) * HB * 64 * sizeof(v4s);
    hipLaunchKernelGGL(k_net_in<HB>, grid, dim3(NB), lds, s, X, f_in, params[0], params[1], keep ? zs : nullptr, hs, n);
    for (int l = 0; l < L; ++l) {
        const bool last = (l == L - 1);
        const float* h = hs + (keep ? l : l & 1) * row;
        float* hn = keep ? hs + (l + 1) * row : last ? nullptr : hs + ((l + 1) & 1) * row;
        hipLaunchKernelGGL(k_net_layer<HB>, grid, dim3(NB), 0, s, h, ptr, idx, params[2 + 2 * l], params[3 + 2 * l],
                           keep ? as + l * row : nullptr, keep ? zs + (l + 1) * row : nullptr, hn, params[2 * L + 2],
                           params[2 * L + 3], last ? y : nullptr, f_out, n);
    }
}

template <int HB>
void net_backward(const float* const* params, int f_in, int f_out, int L, const float* X, const int32_t* ptr,
                  const int32_t* idx, int n, const float* cache, int cache_n, const float* dY, float* const* grads,
                  float* ws, hipStream_t s) {
    constexpr int H = 16 * HB;
    const size_t crow = (size_t)cache_n * H, row = (size_t)n * H;
    const float* const hs = cache;
    const float* const zs = cache + (L + 1) * crow;
    const float* const as = zs + (L + 1) * crow;
    float* const dzs = ws;
    float* const dH = dzs + (L + 1) * row;
    float* const Gs[2] = {dH + row, dH + 2 * row};
    float* part = dH + 3 * row;
    const dim3 grid(net_blocks(n));
    for (int l = L; l >= 0; --l) {
        // layer l of the cache: z_l = the argument of silu, W of the layer that made it
        hipLaunchKernelGGL(k_net_layer_bwd<HB>, grid, dim3(NB), 0, s, l == L ? dY : nullptr, params[2 * L + 2], f_out, dH,
                           l < L ? (const float*)Gs[(l + 1) & 1] : nullptr, ptr, idx, zs + l * crow,
                           l > 0 ? params[2 * l] : nullptr, dzs + l * row, Gs[l & 1], n);
    }
    WArgs w;
    FinalArgs f;
    w.nodes = n;
    w.kchunk = node_chunk(n);
    w.splits = node_splits(n);
    w.parts = (n + COL_ROWS - 1) / COL_ROWS;
    w.sum_blocks = (w.parts + NW - 1) / NW;
    w.n_probs = w.n_sums = w.m_blocks = f.n_segs = 0;
    int seg_blocks = 0;
    auto segment = [&](const float* src, float* out, int len, int parts) {
        f.s[f.n_segs++] = FinalSeg{src, out, len, parts, seg_blocks};
        seg_blocks += (len + 63) / 64;
    };
    auto product = [&](const float* A, int m, const float* B, int nc, float* out) {
        w.p[w.n_probs++] = WProb{A, B, w.splits > 1 ? part : out, m, nc, w.m_blocks};
        w.m_blocks += ((m + WM - 1) / WM) * ((nc + WN - 1) / WN);
        if (w.splits > 1) {
            segment(part, out, m * nc, w.splits);
            part += (size_t)w.splits * m * nc;
        }
    };
    auto colsum = [&](const float* B, int nc, float* out) {
        w.c[w.n_sums++] = WColsum{B, part, nc};
        segment(part, out, nc, w.parts);
        part += (size_t)w.parts * nc;
    };
    for (int l = L; l > 0; --l) {
        product(hs + (l - 1) * crow, H, dzs + l * row, H, grads[2 * l]);
        product(as + (l - 1) * crow, H, dzs + l * row, H, grads[2 * l] + H * H);
        colsum(dzs + l * row, H, grads[2 * l + 1]);
    }
    product(X, f_in, dzs, H, grads[0]);
    colsum(dzs, H, grads[1]);
    product(hs + L * crow, H, dY, f_out, grads[2 * L + 2]);
    colsum(dY, f_out, grads[2 * L + 3]);
    const int nb = w.n_sums * w.sum_blocks + (w.m_blocks * w.splits + 7) / 8 * 8;
    hipLaunchKernelGGL(k_net_wgrad, dim3(nb), dim3(NB), 0, s, w);
    hipLaunchKernelGGL(k_net_sums, dim3(seg_blocks), dim3(64), 0, s, f);
}

}  // namespace

extern "C" {

int bt_gnn_gemm(const float* A, int64_t sam, int64_t sak, const float* B, int64_t sbk, int64_t sbn,
                float* C, int64_t ldc, int32_t m, int32_t n, int32_t k, int32_t beta,
                float* ws, int32_t ksplit, void* stream) {
    if (!A || !B || !C || m < 1 || n < 1 || k < 1 || ksplit < 1) return BT_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    if (ksplit > 1 && !ws) return BT_EINVAL;
    int kchunk = (k + ksplit - 1) / ksplit;
    kchunk = (kchunk + 15) / 16 * 16;
    const int splits = (k + kchunk - 1) / kchunk;
    dim3 grid((m + 15) / 16, (n + 63) / 64, splits);
    if (splits == 1 && !beta) {
        hipLaunchKernelGGL(k_gemm_bf16, grid, dim3(256), 0, s, A, (long long)sam, (long long)sak, B,
                           (long long)sbk, (long long)sbn, C, (long long)ldc, m, n, k, kchunk);
    } else {
        if (!ws) return BT_EINVAL;
        hipLaunchKernelGGL(k_gemm_bf16, grid, dim3(256), 0, s, A, (long long)sam, (long long)sak, B,
                           (long long)sbk, (long long)sbn, ws, (long long)n, m, n, k, kchunk);
        hipLaunchKernelGGL(k_sum_splits, dim3(blocks((long long)m * n)), dim3(EB), 0, s,
                           (const float*)ws, splits, C, (long long)ldc, m, n, beta);
    }
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

int bt_gnn_bias_silu(float* Z, const float* b, float* H, const float* Hres, int32_t n, int32_t f, void* stream) {
    if (!Z || !b || !H || n < 1 || f < 1) return BT_EINVAL;
    hipLaunchKernelGGL(k_bias_silu, dim3(blocks((long long)n * f)), dim3(EB), 0, (hipStream_t)stream,
                       Z, b, H, Hres, n, f);
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

int bt_gnn_bias(float* Y, const float* b, int32_t n, int32_t f, void* stream) {
    if (!Y || !b || n < 1 || f < 1) return BT_EINVAL;
    hipLaunchKernelGGL(k_bias, dim3(blocks((long long)n * f)), dim3(EB), 0, (hipStream_t)stream, Y, b, n, f);
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

int bt_gnn_silu_bwd(const float* dH, const float* Z, float* dZ, int64_t count, void* stream) {
    if (!dH || !Z || !dZ || count < 1) return BT_EINVAL;
    hipLaunchKernelGGL(k_silu_bwd, dim3(blocks(count)), dim3(EB), 0, (hipStream_t)stream, dH, Z, dZ,
                       (long long)count);
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

int bt_gnn_mean_agg(const float* H, int64_t ldh, const int32_t* ptr, const int32_t* idx, float* out, int64_t ldo,
                    int32_t n, int32_t f, void* stream) {
    if (!H || !ptr || !idx || !out || n < 1 || f < 1) return BT_EINVAL;
    hipLaunchKernelGGL(k_mean_agg, dim3(blocks((long long)n * f)), dim3(EB), 0, (hipStream_t)stream,
                       H, (long long)ldh, ptr, idx, out, (long long)ldo, n, f);
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

int bt_gnn_mean_agg_T(const float* G, int64_t ldg, const int32_t* ptr, const int32_t* idx, float* out,
                      int64_t ldo, int32_t n, int32_t f, int32_t accumulate, void* stream) {
    if (!G || !ptr || !idx || !out || n < 1 || f < 1) return BT_EINVAL;
    hipLaunchKernelGGL(k_mean_agg_T, dim3(blocks((long long)n * f)), dim3(EB), 0, (hipStream_t)stream,
                       G, (long long)ldg, ptr, idx, out, (long long)ldo, n, f, accumulate);
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

int bt_gnn_colsum(const float* G, int64_t ldg, int32_t n, int32_t f, float* out, float* ws, int32_t ws_len,
                  void* stream) {
    if (!G || !out || !ws || n < 1 || f < 1 || f > EB) return BT_EINVAL;
    const int rpb = colsum_rows_per_block(n, f, ws_len);
    const int parts = (n + rpb - 1) / rpb;
    hipLaunchKernelGGL(k_colsum_part, dim3(parts), dim3(EB), 0, (hipStream_t)stream, G, (long long)ldg, n, f,
                       rpb, ws);
    hipLaunchKernelGGL(k_colsum_final, dim3((f + EB - 1) / EB), dim3(EB), 0, (hipStream_t)stream,
                       (const float*)ws, parts, f, out);
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

int bt_gnn_colsum_noalloc(const float* G, int64_t ldg, int32_t n, int32_t f, float* out, void* stream) {
    if (!G || !out || n < 1 || f < 1) return BT_EINVAL;
    if (f > EB) return BT_EINVAL;          // at most 256 columns (one block of the final sum)
    float* ws = nullptr;
    const int rc = scratch_address(&ws);
    if (rc != BT_OK) return rc;
    // the same launches as bt_gnn_colsum with ws = scratch: every partial is
    // written before it is read, so nothing needs clearing between calls
    const int rpb = colsum_rows_per_block(n, f, BT_GNN_SCRATCH_FLOATS);
    const int parts = (n + rpb - 1) / rpb;
    hipLaunchKernelGGL(k_colsum_part, dim3(parts), dim3(EB), 0, (hipStream_t)stream, G, (long long)ldg, n, f,
                       rpb, ws);
    hipLaunchKernelGGL(k_colsum_final, dim3((f + EB - 1) / EB), dim3(EB), 0, (hipStream_t)stream,
                       (const float*)ws, parts, f, out);
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

int bt_gnn_mse(const float* Y, const float* T, const float* mask, int64_t count, float inv_n, float* dY,
               float* part, int32_t part_len, void* stream) {
    if (!Y || !T || !mask || !dY || !part || count < 1) return BT_EINVAL;
    if ((long long)blocks(count) > part_len) return BT_EINVAL;
    hipLaunchKernelGGL(k_mse, dim3(blocks(count)), dim3(EB), 0, (hipStream_t)stream, Y, T, mask,
                       (long long)count, inv_n, dY, part);
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

int bt_gnn_adam_all(float* const* p, const float* const* g, float* const* m, float* const* v, const int64_t* counts,
                    int32_t n_tensors, float lr, float b1, float b2, float eps, int32_t t, void* stream) {
    if (!p || !g || !m || !v || !counts || n_tensors < 1 || t < 1) return BT_EINVAL;
    for (int q = 0; q < n_tensors; ++q)
        if (!p[q] || !g[q] || !m[q] || !v[q] || counts[q] < 1) return BT_EINVAL;
    AdamArgs a;
    a.lr = lr;
    a.b1 = b1;
    a.b2 = b2;
    a.eps = eps;
    a.c1 = 1.f - powf(b1, (float)t);
    a.c2 = 1.f - powf(b2, (float)t);
    for (int q0 = 0; q0 < n_tensors; q0 += MAX_TENSORS) {
        a.n = std::min(n_tensors - q0, MAX_TENSORS);
        unsigned nb = 0;
        for (int q = 0; q < a.n; ++q) {
            a.p[q] = p[q0 + q];
            a.g[q] = g[q0 + q];
            a.m[q] = m[q0 + q];
            a.v[q] = v[q0 + q];
            a.count[q] = counts[q0 + q];
            a.first[q] = (int)nb;
            nb += blocks(a.count[q]);
        }
        hipLaunchKernelGGL(k_adam, dim3(nb), dim3(EB), 0, (hipStream_t)stream, a);
    }
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

int bt_gnn_adam(float* p, const float* g, float* m, float* v, int64_t count, float lr, float b1, float b2,
                float eps, int32_t t, void* stream) {
    return bt_gnn_adam_all(&p, &g, &m, &v, &count, 1, lr, b1, b2, eps, t, stream);
}

int bt_gnn_layered(int32_t f_in, int32_t f_out, int32_t hidden, int32_t n_layers) {
    return layered(f_in, f_out, hidden, n_layers) ? 1 : 0;
}

int64_t bt_gnn_cache_len(int32_t hidden, int32_t n_layers, int32_t n, int32_t keep) {
    return (int64_t)n * hidden * (keep ? 3 * (int64_t)n_layers + 2 : 2);
}

int64_t bt_gnn_backward_len(int32_t f_in, int32_t f_out, int32_t hidden, int32_t n_layers, int32_t n) {
    if (n < 1) return 0;                                        // (bt_gnn_backward refuses it)
    int64_t len = (int64_t)n * hidden * (n_layers + 4);         // dz of every layer, dH, two of G
    const int64_t H = hidden;
    const int64_t sums = (n + COL_ROWS - 1) / COL_ROWS;
    len += (int64_t)node_splits(n) * (f_in * H + 2 * n_layers * H * H + H * f_out) + sums * (H * (n_layers + 1) + f_out);
    return len;
}

int bt_gnn_forward(const float* const* params, int32_t f_in, int32_t f_out, int32_t hidden, int32_t n_layers,
                   const float* X, const int32_t* ptr, const int32_t* idx, int32_t n, float* cache, int32_t keep,
                   float* y, void* stream) {
    if (!layered(f_in, f_out, hidden, n_layers) || !params || !X || !ptr || !idx || !cache || !y || n < 1 ||
        (int64_t)n * hidden >= MAX_FLOATS ||
        ((uintptr_t)cache & 15))
        return BT_EINVAL;
    for (int q = 0; q < 2 * n_layers + 4; ++q)
        if (!params[q]) return BT_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    switch (hidden) {
        case 16: net_forward<1>(params, f_in, f_out, n_layers, X, ptr, idx, n, cache, keep != 0, y, s); break;
        case 32: net_forward<2>(params, f_in, f_out, n_layers, X, ptr, idx, n, cache, keep != 0, y, s); break;
        case 64: net_forward<4>(params, f_in, f_out, n_layers, X, ptr, idx, n, cache, keep != 0, y, s); break;
        default: return BT_EINVAL;
    }
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

int bt_gnn_backward(const float* const* params, int32_t f_in, int32_t f_out, int32_t hidden, int32_t n_layers,
                    const float* X, const int32_t* ptr, const int32_t* idx, int32_t n, const float* cache,
                    int32_t cache_n, const float* dY, float* const* grads, float* ws, int64_t ws_len, void* stream) {
    if (!layered(f_in, f_out, hidden, n_layers) || !params || !X || !ptr || !idx || !cache || !dY || !grads || !ws ||
        n < 1 || cache_n < n || (int64_t)cache_n * hidden >= MAX_FLOATS || ((uintptr_t)cache & 15) || ((uintptr_t)ws & 15) || ws_len < bt_gnn_backward_len(f_in, f_out, hidden, n_layers, n))
        return BT_EINVAL;
    for (int q = 0; q < 2 * n_layers + 4; ++q)
        if (!params[q] || !grads[q]) return BT_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    switch (hidden) {
        case 16: net_backward<1>(params, f_in, f_out, n_layers, X, ptr, idx, n, cache, cache_n, dY, grads, ws, s); break;
        case 32: net_backward<2>(params, f_in, f_out, n_layers, X, ptr, idx, n, cache, cache_n, dY, grads, ws, s); break;
        case 64: net_backward<4>(params, f_in, f_out, n_layers, X, ptr, idx, n, cache, cache_n, dY, grads, ws, s); break;
        default: return BT_EINVAL;
    }
    return hipGetLastError() == hipSuccess ? BT_OK : BT_EHIP;
}

}  // extern "C"
