// Kernels around the GEMM: bias, ReLU forward/backward, column sums, the MLP
// step's head, SGD and the Philox random fills (row softmax and softmax
// cross-entropy are in row_kernels.hip).  All are HBM- or latency-bound; none uses
// atomics, so every result is deterministic run to run.
#include "fdl_device.hpp"
#include "fdl_internal.hpp"

#include <algorithm>

namespace fdl {

namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(int64_t n, int per_thread = 1) {
    const int64_t threads = (n + per_thread - 1) / per_thread;
    const int64_t blocks = (threads + kBlock - 1) / kBlock;
    return (unsigned)std::min<int64_t>(blocks, 1 << 20);
}

// dst[e] = src[e] for e < n by a block of kBlock threads, 16 loads in flight
// per thread before their LDS stores (a plain strided loop waits out one
// global-memory round trip per iteration).
__device__ __forceinline__ void stage_to_lds(float* __restrict__ dst, const float* __restrict__ src,
                                             int n) {
    constexpr int kBatch = 16;
    const int t = threadIdx.x;
    for (int e0 = 0; e0 < n; e0 += kBatch * kBlock) {
        float v[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int e = e0 + u * kBlock + t;
            v[u] = e < n ? src[e] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int e = e0 + u * kBlock + t;
            if (e < n) dst[e] = v[u];
        }
    }
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Column sums of a tall matrix.  No block can add another's partial sums
// without scratch memory, so each column is summed by one block and the
// parallelism is across columns: strips of kTallCols columns (one 16-byte load
// per row where rows are 16-byte aligned), 1024 threads of a block on 1024 rows at once, kUnroll rows
// in flight each.  What bounds it is the cache lines a CU can take in, about
// one per nanosecond whatever the width of the strip, so narrow strips on many
// CUs win; the blocks whose strips share a 128-byte line are numbered onto one
// XCD, whose L2 then fetches the line once (without that 60000 x 256 took 122
// us, as eight fetches of everything).  60000 x 256: 148 -> 55 us, 60000 x 1024:
// 151 -> 98 us, 4096 x 512: 8.0 -> 6.3 us; wider strips (8, 16 and 32
// columns) 99, 107 and 112 us at 60000 x 256.
constexpr int kTallThreads = 1024;
constexpr int kTallCols = 4;

// Whether rows of `cols` floats from x take 16-byte loads.
inline bool vec_rows(const float* x, int64_t cols) {
    return cols % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
}

// Whether the strips beat colsum_kernel's 32-column blocks, which read whole
// lines but leave CUs idle below 8192 columns.  Measured (us, blocks / strips):
// * Up to 2048 rows the blocks' one round trip wins (1024 x 256 2.9 / 3.1).
// * Up to 1024 columns every strip has a CU of its own: 4096 x 1000 13.3 / 7.9,
//   30000 x 512 76 / 41; only wide matrices of few rows lose (2049 x 1024
//   5.2 / 5.6, 2500 x 1024 6.0 / 6.0).
// * Up to 2048 columns a CU has two.  Blocks whose columns straddle lines lose
//   still (4096 x 1500 15.3 / 12.1, 8192 x 2000 25.3 / 24.3), aligned ones win
//   until their few CUs are the bound (4096 x 2048 9.2 / 11.8, 8192 x 2048
//   22.6 / 24.4, 16384 x 1536 42.6 / 42.1, 60000 x 2048 263 / 241).
// * Beyond, the strips' partial lines are the bound (4096 x 8192 22.5 / 40.4,
//   60000 x 4096 266 / 522, 8192 x 2200 26.3 / 31.7).
// * With 4-byte loads the strips win where the rows' alignment varies and there
//   are enough of them (4096 x 1001 15.6 / 9.2, 8192 x 333 25.5 / 12.9, 4096 x 10
//   7.6 / 6.2, but 2049 x 333 5.1 / 5.9, 60000 x 1501 251 / 255), and lose where
//   it does not (4096 x 512 one float off 7.8 / 10.2, 60000 x 1024 211 / 273).
inline bool tall_strips(const float* x, int64_t rows, int64_t cols) {
    if (rows <= 2048 || cols > 2048) return false;
    if (!vec_rows(x, cols)) {
        return cols % 8 != 0 && cols <= 1024 && (cols <= 128 || rows >= 3000);
    }
    if (cols <= 768) return true;
    const bool whole_lines = cols % 32 == 0 && (reinterpret_cast<uintptr_t>(x) & 127u) == 0;
    if (!whole_lines) return true;
    return rows >= (cols <= 1024 ? 2500 : 16384);
}

template <bool VEC>
__device__ __forceinline__ void colsum_tall_body(const float* __restrict__ x,
                                                 float* __restrict__ out,
                                                 float* __restrict__ param, float lr,
                                                 int64_t rows, int64_t cols, int block,
                                                 int nblocks) {
#pragma clang fp contract(off)
    constexpr int V = kTallCols, kUnroll = 4;
    constexpr int kWaves = kTallThreads / 64;
    __shared__ float red[kWaves][V];
    // strips in order over XCDs (block b runs on XCD b % 8), each a contiguous range
    const int64_t per = nblocks / 8, extra = nblocks % 8;
    const int64_t xcd = block % 8;
    const int64_t c0 = (xcd * per + min(xcd, extra) + block / 8) * V;
    const float* col = x + c0;
    float s[V] = {};
    for (int64_t r0 = threadIdx.x; r0 < rows; r0 += (int64_t)kUnroll * kTallThreads) {
        float q[kUnroll][V];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const float* p = col + min(r0 + u * (int64_t)kTallThreads, rows - 1) * cols;
            if constexpr (VEC) {
                const floatx4 z = *reinterpret_cast<const floatx4*>(p);
#pragma unroll
                for (int v = 0; v < V; ++v) q[u][v] = z[v];
            } else {
#pragma unroll
                for (int v = 0; v < V; ++v) q[u][v] = p[min((int64_t)v, cols - 1 - c0)];
            }
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
#pragma unroll
            for (int v = 0; v < V; ++v)
                s[v] += r0 + u * (int64_t)kTallThreads < rows ? q[u][v] : 0.0f;
    }
    // lanes by a fixed exchange tree, then the waves in order
#pragma unroll
    for (int v = 0; v < V; ++v) {
        s[v] = wave_sum(s[v]);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64][v] = s[v];
    }
    __syncthreads();
    const int64_t c = c0 + threadIdx.x;
    if (threadIdx.x < V && c < cols) {
        float t = red[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) t += red[w][threadIdx.x];
        out[c] = t;
        if (param) {
            const float step = lr * t;
            param[c] -= step;
        }
    }
}

template <bool VEC>
__global__ void __launch_bounds__(kTallThreads)
colsum_tall_kernel(const float* __restrict__ x, float* __restrict__ out,
                   float* __restrict__ param, float lr, int64_t rows, int64_t cols) {
    colsum_tall_body<VEC>(x, out, param, lr, rows, cols, blockIdx.x, gridDim.x);
}

// The reductions of a large training step in one launch: db1 and db2, the
// column sums of G1 (blocks 0 .. n1 - 1) and of G2 (the next n2), and the loss, the sum of
// nparts partial sums `stride` floats apart (the last block).  n1 or n2 may be
// 0: that sum has a launch of its own.
template <bool VEC1, bool VEC2>
__global__ void __launch_bounds__(kTallThreads)
step_reduce_kernel(const float* __restrict__ G1, float* __restrict__ db1, int hidden, int n1,
                   const float* __restrict__ G2, float* __restrict__ db2, int classes, int n2,
                   int64_t rows, const float* __restrict__ part, int nparts, int stride,
                   float* __restrict__ loss) {
    const int block = blockIdx.x;
    if (block < n1) {
        colsum_tall_body<VEC1>(G1, db1, nullptr, 0.0f, rows, hidden, block, n1);
    } else if (block < n1 + n2) {
        colsum_tall_body<VEC2>(G2, db2, nullptr, 0.0f, rows, classes, block - n1, n2);
    } else {
        constexpr int kWaves = kTallThreads / 64;
        __shared__ float red[kWaves];
        float s = 0.0f;
        for (int b = threadIdx.x; b < nparts; b += kTallThreads) s += part[(int64_t)b * stride];
        s = wave_sum(s);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64] = s;
        __syncthreads();
        if (threadIdx.x == 0) {
            float t = red[0];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) t += red[w];
            loss[0] = t;
        }
    }
}

// out[r, c] += bias[c]   (src/kernels/cuda/bias.cu:5-12 semantics)
__global__ void add_row_bias_kernel(float* __restrict__ out,
                                    const float* __restrict__ bias,
                                    int64_t rows, int64_t cols) {
    const int64_t n = rows * cols;
    for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < n;
         idx += (int64_t)gridDim.x * blockDim.x) {
        out[idx] += bias[idx % cols];
    }
}

// out[i] = op(a[i], b[i]) over n floats.  HBM-bound: 16 bytes per lane and
// access where every operand is 16-byte aligned (`out` may be `a` or `b`), one
// float per lane otherwise and for the last n % 4.  Outputs of kStreamBytes, the
// Infinity Cache's size, or more leave through non-temporal stores (2^26 floats:
// relu 91 -> 79 us, with a pass over its output 178 -> 173, with a product
// that reads it 315 -> 321); of smaller ones a part is still there when the
// reader comes (60000 x 256: relu and a pass over its output 38.4 us, 42.7
// with non-temporal stores).  15.4M floats: relu 25.8 -> 19.3 us (6.4 TB/s),
// relu_backward 36.3 -> 27.2 us (6.8 TB/s).  More than one access per thread
// was no faster (2, 4 and 8: within 3%).
struct OpRelu {
    static constexpr bool kTwo = false;
    float lr;
    __device__ __forceinline__ float operator()(float a, float) const { return fmaxf(0.0f, a); }
};
struct OpReluBackward {
    static constexpr bool kTwo = true;
    float lr;
    __device__ __forceinline__ float operator()(float g, float act) const {
        return act > 0.0f ? g : 0.0f;
    }
};
// The product is rounded before the subtraction (no FMA contraction), as the
// reference's x86 host update computes it.
struct OpSgd {
    static constexpr bool kTwo = true;
    float lr;
    __device__ __forceinline__ float operator()(float p, float g) const {
#pragma clang fp contract(off)
        const float step = lr * g;
        return p - step;
    }
};

template <class Op, bool VEC, bool NT>
__global__ void __launch_bounds__(kBlock)
elementwise_kernel(const float* a, const float* b, float* out, int64_t n, Op op) {
    const int64_t n4 = n / 4;
    const int64_t units = VEC ? n4 + (n - 4 * n4) : n;
    for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < units;
         i += (int64_t)gridDim.x * kBlock) {
        if (VEC && i < n4) {
            const floatx4 va = reinterpret_cast<const floatx4*>(a)[i];
            floatx4 vb = va;
            if constexpr (Op::kTwo) vb = reinterpret_cast<const floatx4*>(b)[i];
            floatx4 r;
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = op(va[e], vb[e]);
            floatx4* dst = reinterpret_cast<floatx4*>(out) + i;
            if constexpr (NT) {
                __builtin_nontemporal_store(r, dst);
            } else {
                *dst = r;
            }
        } else {
            const int64_t e = VEC ? i + 3 * n4 : i;  // the last n % 4 floats follow the n4 units
            out[e] = op(a[e], Op::kTwo ? b[e] : 0.0f);
        }
    }
}

constexpr int64_t kStreamBytes = int64_t(256) << 20;

template <class Op>
hipError_t launch_elementwise(const float* a, const float* b, float* out, int64_t n, Op op,
                              bool streams, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    const bool vec = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) |
                       reinterpret_cast<uintptr_t>(out)) & 15u) == 0;
    // (4 bytes per lane: four accesses per thread; with one each 2^23 floats one
    // float off took sgd 19.1 us against 17.3, relu 16.1 against 12.8)
    const dim3 grid(vec ? grid_for(n / 4 + n % 4) : grid_for(n, 4));
    if (!vec) {
        hipLaunchKernelGGL((elementwise_kernel<Op, false, false>), grid, dim3(kBlock), 0, stream,
                           a, b, out, n, op);
    } else if (streams && n * (int64_t)sizeof(float) >= kStreamBytes) {
        hipLaunchKernelGGL((elementwise_kernel<Op, true, true>), grid, dim3(kBlock), 0, stream, a,
                           b, out, n, op);
    } else {
        hipLaunchKernelGGL((elementwise_kernel<Op, true, false>), grid, dim3(kBlock), 0, stream,
                           a, b, out, n, op);
    }
    return hipGetLastError();
}

__global__ void __launch_bounds__(kColsumThreads)
colsum_kernel(const float* __restrict__ x, float* __restrict__ out,
              float* __restrict__ param, float lr, int64_t rows, int64_t cols) {
    colsum_body(x, out, param, lr, rows, cols, blockIdx.x);
}

// Softmax cross-entropy for classes <= kXentFusedMaxClasses with the bias
// gradient and the bias SGD step fused: one block walks the batch in chunks of
// 256 rows staged through LDS with coalesced loads (thread t owns row t of
// the chunk), writes the gradient through LDS with coalesced stores, and adds
// each chunk's gradient column sums in row order.  db and bparam are written
// once at the end.
__global__ void __launch_bounds__(kBlock)
softmax_xent_db_sgd_kernel(const float* __restrict__ logits,
                           const int64_t* __restrict__ labels, float* __restrict__ loss,
                           float* __restrict__ grad, float* __restrict__ db,
                           float* __restrict__ bparam, float lr, int64_t batch,
                           int64_t classes) {
#pragma clang fp contract(off)
    __shared__ float zs[kBlock * kXentFusedMaxClasses];
    __shared__ float part[kBlock];
    __shared__ float wpart[kBlock / 64];
    const int t = threadIdx.x;
    const float inv_b = 1.0f / (float)batch;
    // Loads whose values are needed late are issued first, so the step pays
    // one global-memory round trip, not one per phase.
    const float bold = t < classes ? bparam[t] : 0.0f;
    float lsum = 0.0f;
    // Column sums of the gradient: thread t adds class cls over the rows
    // r = grp, grp + ngrp, ... of each chunk (ngrp groups of cpad threads).
    const int cpad = classes <= 8 ? 8 : (classes <= 16 ? 16 : 32);
    const int ngrp = kBlock / cpad;
    const int cls = t % cpad;
    const int grp = t / cpad;
    float dbc = 0.0f;
    for (int64_t r0 = 0; r0 < batch; r0 += kBlock) {
        const int rows = (int)min<int64_t>(kBlock, batch - r0);
        const int n = rows * (int)classes;
        const int64_t label = t < rows ? labels[r0 + t] : -1;
        stage_to_lds(zs, logits + r0 * classes, n);
        __syncthreads();
        if (t < rows) {
            float* z = zs + t * classes;
            float mx = z[0];
            for (int c = 1; c < classes; ++c) mx = fmaxf(mx, z[c]);
            float s = 0.0f;
            for (int c = 0; c < classes; ++c) s += expf(z[c] - mx);
            const bool valid = label >= 0 && label < classes;
            if (valid) lsum += (logf(s) + mx - z[label]) * inv_b;
            const float inv_s = 1.0f / s;
            for (int c = 0; c < classes; ++c) {
                float pc = expf(z[c] - mx) * inv_s;
                if (valid && c == label) pc -= 1.0f;
                z[c] = pc * inv_b;
            }
        }
        __syncthreads();
        float* gdst = grad + r0 * classes;
        for (int e = t; e < n; e += kBlock) gdst[e] = zs[e];
        if (cls < classes) {
            for (int r = grp; r < rows; r += ngrp) dbc += zs[r * classes + cls];
        }
        __syncthreads();
    }
    // Group partials of each class, added in group order; the loss is summed
    // within each wave, then over the waves in wave order.
    part[t] = dbc;
    lsum = wave_sum(lsum);
    if ((t & 63) == 0) wpart[t >> 6] = lsum;
    __syncthreads();
    if (t < classes) {
        float d = part[t];
        for (int g = 1; g < ngrp; ++g) d += part[g * cpad + t];
        db[t] = d;
        const float step = lr * d;
        bparam[t] = bold - step;
    }
    if (t == 0 && loss) {
        float l = wpart[0];
        for (int w = 1; w < kBlock / 64; ++w) l += wpart[w];
        loss[0] = l;
    }
}

// The MLP step's head: kHeadRows rows per block, one half-wave (32 lanes) per
// row; CM >= classes and 32 * NH >= hidden are compile-time bounds.  Lane l
// holds H[row][l + 32 k].  W2 is staged in LDS as 32 * NH rows of CM floats
// (row stride CM + 4), zero past `hidden` rows and `classes` columns, so every loop over classes
// runs to CM with no bounds test (the padding adds exact zeros) and its LDS
// reads are issued together.
//   logits[row][c] = sum_j H[row][j] W2[j][c] + b2[c]: the 32 lane partials
//     meet in an xor butterfly, so every lane of the row ends with the same
//     sums; the bias is added after the sum, as in linear_cpu
//     (tests/tensor/linear_tensor_test.cpp:17-25).
//   loss share and G2[row][c] as in softmax_xent_db_sgd_kernel (the legacy
//     SoftmaxCrossEntropyLoss forward and backward,
//     legacy/src/ops/SoftmaxCrossEntropyLoss.cpp:39-51).
//   G1[row][j] = H[row][j] > 0 ? sum_c G2[row][c] W2[j][c] : 0 (the NT product
//     dY1 = G2 W2^T of legacy/src/ops/Layers.cpp:36 through the ReLU mask).
// The block's record at part + block * (classes + 1): the column sums of its
// G2 rows (rows in order), then the sum of its rows' loss shares;
// xent_finalize_body adds the records in block order.
__device__ __forceinline__ float half_wave_max(float x) {
    x = fmaxf(x, half_wave_partner<0>(x));
    x = fmaxf(x, half_wave_partner<1>(x));
    x = fmaxf(x, half_wave_partner<2>(x));
    x = fmaxf(x, half_wave_partner<3>(x));
    return fmaxf(x, half_wave_partner<4>(x));
}

__device__ __forceinline__ float half_wave_sum(float x) {
    x += half_wave_partner<0>(x);
    x += half_wave_partner<1>(x);
    x += half_wave_partner<2>(x);
    x += half_wave_partner<3>(x);
    return x + half_wave_partner<4>(x);
}

// One step of the transposing reduction: each lane holds N partial sums
// (one per class of its current set); it keeps the lower or upper half of
// the set (by the lane bit this step's pairing splits on) and adds the
// partner's partial sums of the same half.  Each lane sends the half its
// partner keeps, so a step costs N/2 exchanges.
template <int kStep, int N>
__device__ __forceinline__ void transpose_step(float (&v)[N], int lane) {
    constexpr int kHalf = N / 2;
    const bool upper = (lane >> (4 - kStep)) & 1;
#pragma unroll
    for (int i = 0; i < kHalf; ++i) {
        const float send = upper ? v[i] : v[kHalf + i];
        const float keep = upper ? v[kHalf + i] : v[i];
        v[i] = keep + half_wave_partner<kStep>(send);
    }
}

// Sums CM per-lane partials over the 32 lanes of a half-wave, class by
// class, leaving each lane with one class's total: class lane & 31 for
// CM = 32, class (lane & 31) >> 1 for CM = 16 (lanes 2c and 2c + 1 hold the
// same total).  31 (or 16) exchanges instead of 5 per class.
template <int CM>
__device__ __forceinline__ float transpose_sum(float (&v)[CM], int lane) {
    static_assert(CM == 16 || CM == 32, "16 or 32 classes");
    if constexpr (CM == 32) {
        transpose_step<0, 32>(v, lane);
        transpose_step<1, 16>(*reinterpret_cast<float(*)[16]>(v), lane);
        transpose_step<2, 8>(*reinterpret_cast<float(*)[8]>(v), lane);
        transpose_step<3, 4>(*reinterpret_cast<float(*)[4]>(v), lane);
        transpose_step<4, 2>(*reinterpret_cast<float(*)[2]>(v), lane);
        return v[0];
    } else {
        transpose_step<0, 16>(v, lane);
        transpose_step<1, 8>(*reinterpret_cast<float(*)[8]>(v), lane);
        transpose_step<2, 4>(*reinterpret_cast<float(*)[4]>(v), lane);
        transpose_step<3, 2>(*reinterpret_cast<float(*)[2]>(v), lane);
        return v[0] + half_wave_partner<4>(v[0]);
    }
}

template <int CM, int NH>
__global__ void __launch_bounds__(kBlock)
mlp_head_kernel(const float* __restrict__ H, const float* __restrict__ W2,
                const float* __restrict__ b2, const int64_t* __restrict__ labels,
                float* __restrict__ logits, float* __restrict__ G2, float* __restrict__ G1,
                float* __restrict__ part, int batch, int hidden, int classes) {
    constexpr int JR = 32 * NH;                  // W2 rows staged
    constexpr int LR = CM + 4;                   // LDS row stride: 16 consecutive lanes
                                                 // read 16-byte pieces on distinct banks
    constexpr int kPerThread = JR * CM / kBlock;  // staged floats per thread
    static_assert(kPerThread % 16 == 0, "staging runs in batches of 16 loads");
    __shared__ __attribute__((aligned(16))) float w2s[JR * LR];
    __shared__ float b2s[CM];
    __shared__ float g2s[kHeadRows][CM];
    __shared__ float ls[kHeadRows];
    const int t = threadIdx.x;
    const int lane = t & 31;
    const int rl = t >> 5;
    const int row = blockIdx.x * kHeadRows + rl;
    const bool live = row < batch;
    const int rowc = live ? row : batch - 1;  // clamped: loads stay in bounds
    // Every global load below is issued unconditionally at an address
    // clamped into its array, and values outside the problem are zeroed by
    // a select after the load: a load under a lane-divergent branch makes
    // the compiler wait for it before issuing the ones after it, which
    // turned the staging into two dependent round trips.
    const int64_t label = labels[rowc];
    const float* hrow = H + (int64_t)rowc * hidden;
    float h[NH];
#pragma unroll
    for (int k = 0; k < NH; ++k) h[k] = hrow[min(lane + 32 * k, hidden - 1)];
    const float b2v = b2[min(t, classes - 1)];
    // W2 in batches of sixteen loads in flight per thread.
#pragma unroll
    for (int b0 = 0; b0 < kPerThread; b0 += 16) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int e = (b0 + u) * kBlock + t;
            const int j = e / CM, c = e % CM;
            v[u] = W2[min(j, hidden - 1) * classes + min(c, classes - 1)];
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int e = (b0 + u) * kBlock + t;
            const int j = e / CM, c = e % CM;
            w2s[j * LR + c] = (j < hidden && c < classes) ? v[u] : 0.0f;
        }
    }
#pragma unroll
    for (int k = 0; k < NH; ++k) h[k] = lane + 32 * k < hidden ? h[k] : 0.0f;
    if (t < CM) b2s[t] = t < classes ? b2v : 0.0f;
    __syncthreads();

    float z[CM];
#pragma unroll
    for (int c = 0; c < CM; ++c) z[c] = 0.0f;
#pragma unroll
    for (int k = 0; k < NH; ++k) {
        const float* w = w2s + (lane + 32 * k) * LR;
#pragma unroll
        for (int c = 0; c < CM; ++c) z[c] = fmaf(h[k], w[c], z[c]);
    }
    // Each lane ends with one class's logit: class c of lane (c for CM = 32,
    // lanes 2c and 2c + 1 for CM = 16).  The softmax runs on that class
    // alone; the row's maximum, exponent sum and label logit are half-wave
    // reductions.  Lanes of padded classes (c >= classes) hold 0 and take
    // no part.
    const int c = CM == 32 ? lane : lane >> 1;
    const bool owner = CM == 32 || (lane & 1) == 0;  // counts class c once
    const bool cls = c < classes;
    float zc = transpose_sum<CM>(z, lane);
    float gc;
    float loss_share = 0.0f;
    {
#pragma clang fp contract(off)
        const float inv_b = 1.0f / (float)batch;
        zc = zc + b2s[c];
        const float mx = half_wave_max(cls ? zc : -INFINITY);
        const float ez = cls ? expf(zc - mx) : 0.0f;
        const float s = half_wave_sum(owner ? ez : 0.0f);
        const bool valid = label >= 0 && label < classes;
        const float zl = half_wave_sum(owner && c == label ? zc : 0.0f);
        if (valid && live) loss_share = (logf(s) + mx - zl) * inv_b;
        const float inv_s = 1.0f / s;
        float pc = cls ? ez * inv_s : 0.0f;
        if (valid && c == label) pc -= 1.0f;
        gc = pc * inv_b;
    }
    if (owner && cls) {
        if (live) {
            logits[(int64_t)row * classes + c] = zc;
            G2[(int64_t)row * classes + c] = gc;
        }
        g2s[rl][c] = live ? gc : 0.0f;
    }
    if (lane == 0) ls[rl] = loss_share;
    if (owner && !cls && c < CM) g2s[rl][c] = 0.0f;  // padded classes of the row
    __syncthreads();

    // G1 = (G2 W2^T) * [H > 0]: the row's G2 comes back from LDS as
    // broadcast reads, summed in class order.
    float g[CM];
#pragma unroll
    for (int q = 0; q < CM; ++q) g[q] = g2s[rl][q];
    float* g1row = G1 + (int64_t)rowc * hidden;
#pragma unroll
    for (int k = 0; k < NH; ++k) {
        const int j = lane + 32 * k;
        const float* w = w2s + j * LR;
        float v = 0.0f;
#pragma unroll
        for (int q = 0; q < CM; ++q) v = fmaf(g[q], w[q], v);
        if (live && j < hidden) g1row[j] = h[k] > 0.0f ? v : 0.0f;
    }
    if (t <= classes) {
#pragma clang fp contract(off)
        float acc = 0.0f;
        if (t < classes) {
#pragma unroll
            for (int r = 0; r < kHeadRows; ++r) acc += g2s[r][t];
        } else {
#pragma unroll
            for (int r = 0; r < kHeadRows; ++r) acc += ls[r];
        }
        part[(int64_t)blockIdx.x * (classes + 1) + t] = acc;
    }
}

// Reductions over the 16 lanes of a DPP row (steps 1 to 4 of the half-wave
// exchanges), leaving the result on every lane of the row.
__device__ __forceinline__ float row16_max(float x) {
    x = fmaxf(x, half_wave_partner<1>(x));
    x = fmaxf(x, half_wave_partner<2>(x));
    x = fmaxf(x, half_wave_partner<3>(x));
    return fmaxf(x, half_wave_partner<4>(x));
}

__device__ __forceinline__ float row16_sum(float x) {
    x += half_wave_partner<1>(x);
    x += half_wave_partner<2>(x);
    x += half_wave_partner<3>(x);
    return x + half_wave_partner<4>(x);
}

// The head fused with dX = G1 W1^T (the NT product of the legacy backward,
// legacy/src/ops/Layers.cpp:36-40), so that the W1 step can share the next
// launch with dW1: dX's last read of W1 is in this launch.  A block takes
// kHdxRows = 16 rows of the batch and kHdxCols = 64 columns of dX; every
// block recomputes the head for its rows and the blocks of column chunk 0
// store logits, G2 and G1.  All three products run on
// v_mfma_f32_16x16x4_f32:
//   operand a: lane l supplies A[i = l % 16][k]
//   operand b: lane l supplies B[k][j = l % 16]
//   result   : lane l, register r holds D[4 * (l / 16) + r][l % 16]
// with the k permutation of the split-K kernels (at step s of a group of 16,
// lane quarter q supplies k0 + 4q + s, so a lane's four values are one
// 16-byte load).
//   z = H W2 (16 rows x CT tiles of 16 classes): wave w adds hidden
//     [32w, 32w + 32) straight from H's rows; the eight waves' tiles meet in
//     LDS and wave 0 adds them in wave order, adds b2 after the sum (as
//     linear_cpu, tests/tensor/linear_tensor_test.cpp:17-25), and takes the
//     softmax of each row over the 16 lanes of a DPP row: G2 as
//     xent_kernel (row_kernels.hip; legacy SoftmaxCrossEntropyLoss,
//     legacy/src/ops/SoftmaxCrossEntropyLoss.cpp:39-51).  The loss is left to
//     head_finalize_body, which reads the stored logits.
//   G1 = (G2 W2^T) * [H > 0] (legacy/src/ops/Layers.cpp:36 through the ReLU
//     mask): wave w makes hidden tiles 2w and 2w + 1, K = the classes.
//   dX = G1 W1^T: wave w makes column tile w % NCT over part w / NCT of the
//     hidden range; the other parts' sums reach part 0's wave through LDS
//     and are added in part order.
// W2 is staged in LDS as rows of CM floats (laid out by head_w2_at), zero
// past `hidden` rows and `classes` columns.  The head's global loads are all
// issued before its first wait, and dX's W1 fragments right after the
// staging barrier (loads complete in order, so the head's waits never count
// them), all at addresses clamped into the arrays; values outside the
// problem are zeroed where they are used.
// Needs hidden <= 256, hidden % 4 == 0, classes <= 16 * CT, and H and W1
// 16-byte aligned (the host checks).
constexpr int kHdxThreads = kHdxRows * 32;
constexpr int kWave = 64;

// LDS layouts of the head, chosen against gfx950's bank rules as measured
// with the LDS bank-conflict counter on single-wave access patterns: a
// 32-bit access is served in two halves of 32 lanes, each free of conflicts
// when its lanes' dword addresses differ mod 32 (equal addresses are free
// for reads); a ds_read_b128 is served in four passes of 16 lanes -- lane l
// in the pass of (l / 32, parity of bits 2..4 of l) -- each free of conflicts
// when its lanes' 16-byte slots differ mod 16.
//
// W2 and G2 tiles of 16 columns (CM == 16): row j sits at 48 j, moved on by
// 16 floats and with its 4-column slots swapped in pairs (XOR 8) when bit 2
// of j is set.  The staging stores (rows j and j + 1 in a half-wave), the z
// reads (rows j and j + 4), the G2 stores (rows r and r + 4) and the G1 b128
// reads (16 rows x 4 slots) are then all free of conflicts.  The shift and
// the swap depend on bit 2 of j alone, so row 4m + s (s < 4) sits s rows
// from row 4m, and adding a multiple of 8 rows or of 16 columns moves an
// address by exactly that many rows and columns: each access below takes a
// per-lane base plus immediate offsets.  Wider tiles keep a padded row of
// CM + 4 floats, for which the same holds.
template <int CM>
__device__ __forceinline__ int head_w2_at(int j, int c) {
    if constexpr (CM == 16) {
        const int b = (j >> 2) & 1;
        return 48 * j + 16 * b + (c ^ (8 * b));
    } else {
        return j * (CM + 4) + c;
    }
}
template <int CM>
constexpr int head_w2_row() { return CM == 16 ? 48 : CM + 4; }

// G1 tile (kHdxRows = 16 rows x 256 hidden, row stride 260): rows whose
// bits 2 and 3 differ swap the 4-column slots of each pair (XOR 4), so the G1
// stores (rows 4q + r of a half-wave, 16 columns each) and the dX b128 reads
// (16 rows, slot q) are both free of conflicts.  The swap depends on r / 4
// alone and touches bit 2 of the column alone, so rows 4q + r (r < 4) and
// columns c + 16k sit r rows and 16k columns from row 4q, column c.
constexpr int kHdxG1Row = 260;
__device__ __forceinline__ int head_g1_at(int r, int c) {
    return r * kHdxG1Row + (c ^ (4 * (((r >> 2) ^ (r >> 3)) & 1)));
}

template <int CT>
__global__ void __launch_bounds__(kHdxThreads)
mlp_head_dx_kernel(int batch, int in_features, int hidden, int classes,
                   const float* __restrict__ H, const float* __restrict__ W2,
                   const float* __restrict__ b2, const int64_t* __restrict__ labels,
                   const float* __restrict__ W1, float* __restrict__ logits,
                   float* __restrict__ G2, float* __restrict__ G1, float* __restrict__ dX) {
    // (the shape and the loaded operands lead the arguments: the first 14
    // dwords arrive preloaded in SGPRs, so the first loads' addresses wait
    // for no scalar load of the rest)
    constexpr int CM = 16 * CT;                  // classes padded to whole tiles
    constexpr int JR = 256;                      // hidden <= JR
    constexpr int LR = head_w2_row<CM>();        // floats per row of w2s and g2s
    constexpr int NW = kHdxThreads / kWave;      // 8 waves
    constexpr int KZ = JR / NW;                  // hidden range of a wave for z
    constexpr int NCT = kHdxCols / 16;           // dX column tiles of a block
    constexpr int NKS = NW / NCT;                // hidden range split in NKS parts
    constexpr int KH = JR / NKS;                 // hidden range of a wave for dX
    constexpr int NG = KH / 16;
    constexpr int kPerThread = JR * CM / kHdxThreads;  // W2 floats staged per thread
    static_assert(KZ == 32 && NW == 8, "z takes two groups of 16 per wave");
    static_assert(JR <= kHdxG1Row, "g1s rows hold the hidden range");
    __shared__ __attribute__((aligned(16))) float w2s[JR * LR];
    __shared__ __attribute__((aligned(16))) float g1s[kHdxRows * kHdxG1Row];
    __shared__ __attribute__((aligned(16))) float g2s[kHdxRows * LR];
    __shared__ __attribute__((aligned(16))) floatx4 zred[NW][CT][kWave];
    __shared__ __attribute__((aligned(16))) floatx4 red[NKS - 1][NCT][kWave];
    __shared__ int64_t lbls[kHdxRows];
    __shared__ float b2s[CM];
    const int t = threadIdx.x;
    const int l64 = t & (kWave - 1);
    const int w = __builtin_amdgcn_readfirstlane(t / kWave);
    const int q = l64 >> 4;
    const int i16 = l64 & 15;
    const int chunk = blockIdx.x;
    const int r0 = blockIdx.y * kHdxRows;
    const bool store_head = chunk == 0;

    // ---- loads ----
    // softmax inputs, staged in LDS with W2 (a load used only inside the
    // softmax branch would be issued there, a round trip late)
    const int64_t lab_t = labels[min(r0 + (t & (kHdxRows - 1)), batch - 1)];
    const float b2_t = b2[min(t & (CM - 1), classes - 1)];
    float v[kPerThread];
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) {
        const int e = u * kHdxThreads + t;
        const int j = e / CM, c = e % CM;
        v[u] = W2[min(j, hidden - 1) * classes + min(c, classes - 1)];
    }
    // z operand a: H[r0 + i16][32w + 16g + 4q .. + 3]
    const float* harow = H + (int64_t)min(r0 + i16, batch - 1) * hidden;
    floatx4 ha[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
        ha[g] = *reinterpret_cast<const floatx4*>(harow + min(w * KZ + 16 * g + 4 * q, hidden - 4));
    }
    // G1's mask: H[r0 + 4q + r][16 (2w + tt) + i16]
    float hm[2][4];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            hm[tt][r] = H[(int64_t)min(r0 + 4 * q + r, batch - 1) * hidden +
                          min(16 * (2 * w + tt) + i16, hidden - 1)];
    // dX's column of this lane (its W1 fragments are loaded after the staging
    // barrier, below)
    const int ct4 = w % NCT;
    const int kh = w / NCT;
    const int col = chunk * kHdxCols + ct4 * 16 + i16;
    // element u * kHdxThreads + t is row u * kStageRows + t / CM, column t % CM
    constexpr int kStageRows = kHdxThreads / CM;
    static_assert(kHdxThreads % CM == 0 && kStageRows % 8 == 0, "staging rows step by 8");
    const int stage_at = head_w2_at<CM>(t / CM, t % CM);
#pragma unroll
    for (int u = 0; u < kPerThread; ++u) {
        const int j = u * kStageRows + t / CM, c = t % CM;
        w2s[stage_at + u * kStageRows * LR] = (j < hidden && c < classes) ? v[u] : 0.0f;
    }
    // every thread stores (threads with equal indices store equal values): a
    // store under a branch would pull its load into the branch
    lbls[t & (kHdxRows - 1)] = lab_t;
    b2s[t & (CM - 1)] = (t & (CM - 1)) < classes ? b2_t : 0.0f;
    __syncthreads();
    // dX operand b: W1[col][k0 .. k0 + 3].  Issued after the barrier, where
    // the head's own loads are in: issued at the start with them, these 64 KB
    // per block competed with them (16.52 -> 16.37 us per step), and issued
    // after the z products' barrier they arrived late for dX (16.64 us).
    const float* w1row = W1 + (int64_t)min(col, in_features - 1) * hidden;
    floatx4 wb[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        wb[g] = *reinterpret_cast<const floatx4*>(w1row + min(kh * KH + 16 * g + 4 * q, hidden - 4));
    }

    // ---- z = H W2: this wave's 32 hidden values ----
    const floatx4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    const bool row_in = r0 + i16 < batch;
    const float* zb = w2s + head_w2_at<CM>(4 * q, i16);   // + (k0 + s2) rows, 16 ct columns
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        floatx4 zacc = zero4;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const int k0 = w * KZ + 16 * g;
            const floatx4 a = (row_in && k0 + 4 * q < hidden) ? ha[g] : zero4;
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2) {
                const float b = zb[(k0 + s2) * LR + 16 * ct];
                zacc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s2], b, zacc, 0, 0, 0);
            }
        }
        zred[w][ct][l64] = zacc;
    }
    __syncthreads();

    // ---- softmax and G2: wave r (< 4) takes register r of the tiles, so a
    // lane holds row 4q + r, class 16 ct + i16, and a DPP row of 16 lanes one
    // row of the batch ----
    if (w < 4) {
#pragma clang fp contract(off)
        const int r = w;
        float zc[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            float zz = zred[0][ct][l64][r];
#pragma unroll
            for (int ww = 1; ww < NW; ++ww) zz += zred[ww][ct][l64][r];
            zc[ct] = zz + b2s[16 * ct + i16];
        }
        const int row = r0 + 4 * q + r;
        const bool live = row < batch;
        float* g2row = g2s + head_w2_at<CM>(4 * q, i16) + r * LR;  // + 16 ct columns
        const int64_t label = lbls[4 * q + r];
        const bool valid = label >= 0 && label < classes;
        const float inv_b = 1.0f / (float)batch;
        float mx = -INFINITY;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            if (16 * ct + i16 < classes) mx = fmaxf(mx, zc[ct]);
        }
        mx = row16_max(mx);
        float ez[CT];
        float es = 0.0f;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            ez[ct] = 16 * ct + i16 < classes ? expf(zc[ct] - mx) : 0.0f;
            es += ez[ct];
        }
        const float inv_s = 1.0f / row16_sum(es);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const int c = 16 * ct + i16;
            float pc = ez[ct] * inv_s;
            if (valid && c == label) pc -= 1.0f;
            const float gc = pc * inv_b;
            if (live && store_head && c < classes) {
                logits[(int64_t)row * classes + c] = zc[ct];
                G2[(int64_t)row * classes + c] = gc;
            }
            g2row[16 * ct] = (live && c < classes) ? gc : 0.0f;
        }
    }
    __syncthreads();

    // ---- G1 = (G2 W2^T) * [H > 0]: hidden tiles 2w and 2w + 1 ----
    const int frag_at = head_w2_at<CM>(i16, 4 * q);   // + 16 rows per tile, 16 g columns
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
        const int j = 16 * (2 * w + tt) + i16;
        floatx4 gacc = zero4;
#pragma unroll
        for (int g = 0; g < CT; ++g) {
            const floatx4 a = *reinterpret_cast<const floatx4*>(g2s + frag_at + 16 * g);
            const floatx4 b = *reinterpret_cast<const floatx4*>(w2s + frag_at + 16 * (2 * w + tt) * LR + 16 * g);
#pragma unroll
            for (int s2 = 0; s2 < 4; ++s2) {
                gacc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s2], b[s2], gacc, 0, 0, 0);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = r0 + 4 * q + r;
            const bool keep = row < batch && j < hidden;
            const float g1 = (keep && hm[tt][r] > 0.0f) ? gacc[r] : 0.0f;
            g1s[head_g1_at(4 * q, j) + r * kHdxG1Row] = g1;
            if (keep && store_head) G1[(int64_t)row * hidden + j] = g1;
        }
    }
    __syncthreads();

    // ---- dX tile: 16 rows x 16 columns per wave over its part of the hidden range ----
    floatx4 acc = zero4;
    const float* arow = g1s + head_g1_at(i16, 4 * q) + kh * KH;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const floatx4 a = *reinterpret_cast<const floatx4*>(arow + 16 * g);
        const floatx4 b = kh * KH + 16 * g + 4 * q < hidden ? wb[g] : zero4;
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2) {
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s2], b[s2], acc, 0, 0, 0);
        }
    }
    if (kh > 0) red[kh - 1][ct4][l64] = acc;
    __syncthreads();
    if (kh == 0) {
#pragma unroll
        for (int p = 0; p < NKS - 1; ++p) acc += red[p][ct4][l64];
        if (col < in_features) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int orow = r0 + 4 * q + r;
                if (orow < batch) dX[(int64_t)orow * in_features + col] = acc[r];
            }
        }
    }
}

struct SgdMulti {
    float* p[4];
    const float* g[4];
    int64_t n[4];
};

// blockIdx.y selects the tensor; the x grid strides over the largest one, 16
// bytes per lane over each tensor's aligned body.
__global__ void __launch_bounds__(kBlock) sgd_multi_kernel(SgdMulti args, OpSgd op) {
    const int t = blockIdx.y;
    float* p = args.p[t];
    const float* g = args.g[t];
    const bool vec = ((reinterpret_cast<uintptr_t>(p) | reinterpret_cast<uintptr_t>(g)) & 15u) == 0;
    const int64_t n4 = vec ? args.n[t] / 4 : 0;
    const int64_t first = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    const int64_t step = (int64_t)gridDim.x * kBlock;
    for (int64_t i = first; i < n4; i += step) {
        const floatx4 vp = reinterpret_cast<const floatx4*>(p)[i];
        const floatx4 vg = reinterpret_cast<const floatx4*>(g)[i];
        floatx4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = op(vp[e], vg[e]);
        reinterpret_cast<floatx4*>(p)[i] = r;
    }
    for (int64_t i = 4 * n4 + first; i < args.n[t]; i += step) p[i] = op(p[i], g[i]);
}

// data[0 .. bytes) = 0: 16-byte stores over the aligned body, byte stores at
// the ends.  A kernel rather than hipMemsetAsync, so that a caller may capture
// it into a graph (a captured memset node gave wrong results on replays).
__global__ void zero_fill_kernel(unsigned char* __restrict__ data, int64_t head, int64_t n16,
                                 int64_t tail) {
    const int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    uint4* body = reinterpret_cast<uint4*>(data + head);
    for (int64_t e = i; e < n16; e += stride) body[e] = make_uint4(0u, 0u, 0u, 0u);
    if (i < head) data[i] = 0;
    if (i < tail) data[head + 16 * n16 + i] = 0;
}

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as
// easy as 1, 2, 3", SC'11): counter (i_lo, i_hi, 0, 0), key = seed.
struct Philox4 {
    uint32_t v[4];
};

__device__ __forceinline__ Philox4 philox4x32_10(uint64_t ctr, uint64_t seed) {
    uint32_t c0 = (uint32_t)ctr, c1 = (uint32_t)(ctr >> 32), c2 = 0u, c3 = 0u;
    uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
    constexpr uint32_t kM0 = 0xD2511F53u, kM1 = 0xCD9E8D57u;
    constexpr uint32_t kW0 = 0x9E3779B9u, kW1 = 0xBB67AE85u;
#pragma unroll
    for (int round = 0; round < 10; ++round) {
        const uint32_t hi0 = __umulhi(kM0, c0), lo0 = kM0 * c0;
        const uint32_t hi1 = __umulhi(kM1, c2), lo1 = kM1 * c2;
        const uint32_t n0 = hi1 ^ c1 ^ k0;
        const uint32_t n2 = hi0 ^ c3 ^ k1;
        c0 = n0;
        c1 = lo1;
        c2 = n2;
        c3 = lo0;
        k0 += kW0;
        k1 += kW1;
    }
    Philox4 out;
    out.v[0] = c0;
    out.v[1] = c1;
    out.v[2] = c2;
    out.v[3] = c3;
    return out;
}

// 24 random bits -> (0, 1].
__device__ __forceinline__ float u01_open_closed(uint32_t x) {
    return (float)((x >> 8) + 1u) * (1.0f / 16777216.0f);
}

__global__ void fill_uniform_kernel(float* __restrict__ data, int64_t n, float low,
                                    float high, uint64_t seed) {
    for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < n;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const Philox4 r = philox4x32_10((uint64_t)idx, seed);
        data[idx] = low + u01_open_closed(r.v[0]) * (high - low);
    }
}

// Box-Muller on two uniforms of the same counter.
__global__ void fill_normal_kernel(float* __restrict__ data, int64_t n, float mean,
                                   float stddev, uint64_t seed) {
    for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < n;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const Philox4 r = philox4x32_10((uint64_t)idx, seed);
        const float u1 = u01_open_closed(r.v[0]);
        const float u2 = (float)(r.v[1] >> 8) * (1.0f / 16777216.0f);
        const float z = sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
        data[idx] = mean + stddev * z;
    }
}

}  // namespace

hipError_t launch_add_row_bias(float* out, const float* bias, int64_t rows,
                               int64_t cols, hipStream_t stream) {
    const int64_t n = rows * cols;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(add_row_bias_kernel, dim3(grid_for(n)), dim3(kBlock), 0,
                       stream, out, bias, rows, cols);
    return hipGetLastError();
}

hipError_t launch_relu(const float* in, float* out, int64_t n, hipStream_t stream) {
    return launch_elementwise(in, nullptr, out, n, OpRelu{0.0f}, true, stream);
}

hipError_t launch_relu_backward(const float* g, const float* act, float* out,
                                int64_t n, hipStream_t stream) {
    return launch_elementwise(g, act, out, n, OpReluBackward{0.0f}, true, stream);
}

hipError_t launch_colsum_sgd(const float* x, float* out, float* param, float lr,
                             int64_t rows, int64_t cols, hipStream_t stream) {
    if (cols == 0) return hipSuccess;
    if (tall_strips(x, rows, cols)) {
        const bool vec = vec_rows(x, cols);
        const dim3 grid((unsigned)((cols + kTallCols - 1) / kTallCols));
        if (vec) {
            hipLaunchKernelGGL((colsum_tall_kernel<true>), grid, dim3(kTallThreads), 0, stream, x,
                               out, param, lr, rows, cols);
        } else {
            hipLaunchKernelGGL((colsum_tall_kernel<false>), grid, dim3(kTallThreads), 0, stream,
                               x, out, param, lr, rows, cols);
        }
        return hipGetLastError();
    }
    const unsigned blocks = (unsigned)((cols + kColsumCols - 1) / kColsumCols);
    hipLaunchKernelGGL(colsum_kernel, dim3(blocks), dim3(kColsumThreads), 0,
                       stream, x, out, param, lr, rows, cols);
    return hipGetLastError();
}

hipError_t launch_colsum(const float* x, float* out, int64_t rows, int64_t cols,
                         hipStream_t stream) {
    return launch_colsum_sgd(x, out, nullptr, 0.0f, rows, cols, stream);
}

hipError_t launch_softmax_xent_db_sgd(const float* logits, const int64_t* labels,
                                      float* loss, float* grad, float* db, float* bparam,
                                      float lr, int64_t batch, int64_t classes,
                                      hipStream_t stream) {
    if (classes > kXentFusedMaxClasses || !grad || !db || !bparam) return hipErrorInvalidValue;
    hipLaunchKernelGGL(softmax_xent_db_sgd_kernel, dim3(1), dim3(kBlock), 0, stream, logits,
                       labels, loss, grad, db, bparam, lr, batch, classes);
    return hipGetLastError();
}

template <int CM, int NH>
hipError_t launch_mlp_head_cfg(const float* H, const float* W2, const float* b2,
                               const int64_t* labels, float* logits, float* G2, float* G1,
                               float* part, int64_t batch, int64_t hidden, int64_t classes,
                               hipStream_t stream) {
    hipLaunchKernelGGL((mlp_head_kernel<CM, NH>), dim3((unsigned)head_blocks(batch)),
                       dim3(kBlock), 0, stream, H, W2, b2, labels, logits, G2, G1, part,
                       (int)batch, (int)hidden, (int)classes);
    return hipGetLastError();
}

hipError_t launch_mlp_head(const float* H, const float* W2, const float* b2,
                           const int64_t* labels, float* logits, float* G2, float* G1,
                           float* part, int64_t batch, int64_t hidden, int64_t classes,
                           hipStream_t stream) {
    if (!head_supported(hidden, classes) || batch < 1 || batch > INT32_MAX) {
        return hipErrorInvalidValue;
    }
    if (classes <= 16) {
        return hidden <= 256 ? launch_mlp_head_cfg<16, 8>(H, W2, b2, labels, logits, G2, G1,
                                                          part, batch, hidden, classes, stream)
                             : launch_mlp_head_cfg<16, 32>(H, W2, b2, labels, logits, G2, G1,
                                                           part, batch, hidden, classes, stream);
    }
    return hidden <= 256 ? launch_mlp_head_cfg<32, 8>(H, W2, b2, labels, logits, G2, G1, part,
                                                      batch, hidden, classes, stream)
                         : launch_mlp_head_cfg<32, 16>(H, W2, b2, labels, logits, G2, G1, part,
                                                       batch, hidden, classes, stream);
}

hipError_t launch_mlp_head_dx(const float* H, const float* W2, const float* b2,
                              const int64_t* labels, const float* W1, float* logits, float* G2,
                              float* G1, float* dX, int64_t batch, int64_t in_features,
                              int64_t hidden, int64_t classes, hipStream_t stream) {
    if (!head_dx_supported(batch, in_features, hidden, classes, H, W1)) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((in_features + kHdxCols - 1) / kHdxCols),
                    (unsigned)((batch + kHdxRows - 1) / kHdxRows));
    if (classes <= 16) {
        hipLaunchKernelGGL((mlp_head_dx_kernel<1>), grid, dim3(kHdxThreads), 0, stream,
                           (int)batch, (int)in_features, (int)hidden, (int)classes, H, W2, b2,
                           labels, W1, logits, G2, G1, dX);
    } else {
        hipLaunchKernelGGL((mlp_head_dx_kernel<2>), grid, dim3(kHdxThreads), 0, stream,
                           (int)batch, (int)in_features, (int)hidden, (int)classes, H, W2, b2,
                           labels, W1, logits, G2, G1, dX);
    }
    return hipGetLastError();
}

// (the parameter is read again by the next step's products: ordinary stores)
hipError_t launch_sgd(float* param, const float* grad, float lr, int64_t n,
                      hipStream_t stream) {
    return launch_elementwise(param, grad, param, n, OpSgd{lr}, false, stream);
}

hipError_t launch_sgd_multi(int count, float* const* params,
                            const float* const* grads, const int64_t* sizes,
                            float lr, hipStream_t stream) {
    if (count <= 0 || count > 4) return hipErrorInvalidValue;
    SgdMulti args{};
    int64_t nmax = 0;
    for (int t = 0; t < count; ++t) {
        args.p[t] = params[t];
        args.g[t] = grads[t];
        args.n[t] = sizes[t];
        nmax = std::max(nmax, sizes[t]);
    }
    if (nmax == 0) return hipSuccess;
    hipLaunchKernelGGL(sgd_multi_kernel, dim3(grid_for(nmax, 4), count),
                       dim3(kBlock), 0, stream, args, OpSgd{lr});
    return hipGetLastError();
}

hipError_t launch_step_reduce(const float* G1, float* db1, int64_t hidden, const float* G2,
                              float* db2, int64_t classes, int64_t rows, const float* part,
                              int64_t nparts, int stride, float* loss, hipStream_t stream) {
    // Sums wider than the strips are good for go to launch_colsum (a launch also
    // holds at most 2^32 threads, 2^24 columns in strips).
    constexpr int64_t kMaxCols = 2048;
    const int n1 = hidden <= kMaxCols ? (int)((hidden + kTallCols - 1) / kTallCols) : 0;
    const int n2 = classes <= kMaxCols ? (int)((classes + kTallCols - 1) / kTallCols) : 0;
    if (n1 == 0) {
        const hipError_t err = launch_colsum(G1, db1, rows, hidden, stream);
        if (err != hipSuccess) return err;
    }
    if (n2 == 0) {
        const hipError_t err = launch_colsum(G2, db2, rows, classes, stream);
        if (err != hipSuccess) return err;
    }
    const dim3 grid(n1 + n2 + 1);
#define FDL_STEP_REDUCE(V1, V2)                                                                  \
    hipLaunchKernelGGL((step_reduce_kernel<V1, V2>), grid, dim3(kTallThreads), 0, stream, G1,   \
                       db1, (int)hidden, n1, G2, db2, (int)classes, n2, rows, part, (int)nparts, \
                       stride, loss)
    if (vec_rows(G1, hidden)) {
        if (vec_rows(G2, classes)) FDL_STEP_REDUCE(true, true);
        else FDL_STEP_REDUCE(true, false);
    } else {
        if (vec_rows(G2, classes)) FDL_STEP_REDUCE(false, true);
        else FDL_STEP_REDUCE(false, false);
    }
#undef FDL_STEP_REDUCE
    return hipGetLastError();
}

hipError_t launch_zero_fill(void* data, int64_t bytes, hipStream_t stream) {
    auto* p = static_cast<unsigned char*>(data);
    const int64_t head = std::min<int64_t>((16 - (reinterpret_cast<uintptr_t>(p) & 15u)) & 15u,
                                           bytes);
    const int64_t n16 = (bytes - head) / 16;
    const int64_t tail = bytes - head - 16 * n16;
    hipLaunchKernelGGL(zero_fill_kernel, dim3(std::max(1u, grid_for(n16, 4))), dim3(kBlock), 0,
                       stream, p, head, n16, tail);
    return hipGetLastError();
}

hipError_t launch_fill_uniform(float* data, int64_t n, float low, float high,
                               uint64_t seed, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(fill_uniform_kernel, dim3(grid_for(n, 4)), dim3(kBlock), 0,
                       stream, data, n, low, high, seed);
    return hipGetLastError();
}

hipError_t launch_fill_normal(float* data, int64_t n, float mean, float stddev,
                              uint64_t seed, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(fill_normal_kernel, dim3(grid_for(n, 4)), dim3(kBlock), 0,
                       stream, data, n, mean, stddev, seed);
    return hipGetLastError();
}

}  // namespace fdl
