// Row softmax and softmax cross-entropy (loss and gradient).  HBM-bound for
// large inputs, latency-bound for small ones.  A row is held in the registers
// of a group of G lanes, so it is read once, its maximum and sum are lane
// exchanges, and its outputs are written once.  No atomics and no scratch
// memory: every sum has a fixed order, so results repeat bit for bit.
#include "fdl_device.hpp"
#include "fdl_internal.hpp"

#include <algorithm>

namespace fdl {

namespace {

constexpr int kWaveLanes = 64;
constexpr int kRowThreads = 256;        // threads per block of a many-block launch
constexpr int kOneBlockThreads = 1024;  // threads of a one-block launch
// Blocks of a cross-entropy launch, each leaving one partial loss: 4096 keep a
// wave per row up to 16384 rows of more than 64 columns (8192 x 1500: 1024
// blocks of two rows per wave took 30.7 us for the gradient alone, against
// softmax's 19.8 us for the same bytes).
constexpr int kMaxRowBlocks = 4096;

// Maximum and sum over the G lanes that hold a row, on every lane of the group.
template <int G>
__device__ __forceinline__ float group_max(float x) {
    if constexpr (G == 64) x = fmaxf(x, __shfl_xor(x, 32, 64));
    if constexpr (G >= 32) x = fmaxf(x, half_wave_partner<0>(x));
    if constexpr (G >= 16) {
        x = fmaxf(x, half_wave_partner<1>(x));
        x = fmaxf(x, half_wave_partner<2>(x));
    }
    if constexpr (G >= 4) {
        x = fmaxf(x, half_wave_partner<3>(x));
        x = fmaxf(x, half_wave_partner<4>(x));
    }
    return x;
}

template <int G>
__device__ __forceinline__ float group_sum(float x) {
    if constexpr (G == 64) x += __shfl_xor(x, 32, 64);
    if constexpr (G >= 32) x += half_wave_partner<0>(x);
    if constexpr (G >= 16) {
        x += half_wave_partner<1>(x);
        x += half_wave_partner<2>(x);
    }
    if constexpr (G >= 4) {
        x += half_wave_partner<3>(x);
        x += half_wave_partner<4>(x);
    }
    return x;
}

// Sum over a block (a multiple of 64 threads, at most 1024), on thread 0: each
// wave's lanes by a fixed exchange tree, then the waves' sums by another (one
// after the other, their additions doubled the error of a small batch's loss).
__device__ __forceinline__ float block_sum(float x) {
    __shared__ float wsum[kOneBlockThreads / kWaveLanes];
    x = group_sum<kWaveLanes>(x);
    if ((threadIdx.x & (kWaveLanes - 1)) == 0) wsum[threadIdx.x / kWaveLanes] = x;
    __syncthreads();
    constexpr int kWaves = kOneBlockThreads / kWaveLanes;
    static_assert(kWaves == 16, "one exchange group of 16 lanes");
    return group_sum<kWaves>(threadIdx.x < blockDim.x / kWaveLanes ? wsum[threadIdx.x] : 0.0f);
}

// Thread t's share of `nparts` <= kMaxRowBlocks partial sums, t, t + NT, ...
// in order (a block of NT threads), their loads issued together.
template <int NT>
__device__ __forceinline__ float thread_partials(const float* part, int nparts) {
    constexpr int kRounds = kMaxRowBlocks / NT;
    static_assert(kMaxRowBlocks % NT == 0, "whole rounds of partial sums");
    float v[kRounds];
#pragma unroll
    for (int i = 0; i < kRounds; ++i) {
        v[i] = part[min((int)threadIdx.x + i * NT, nparts - 1)];
    }
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < kRounds; ++i) {
        s += (int)threadIdx.x + i * NT < nparts ? v[i] : 0.0f;
    }
    return s;
}

// One row of at most G * R * V columns in the registers of G lanes: lane l
// holds units l, l + G, ... of V consecutive columns.  Loads are issued
// together at addresses clamped into the row; columns past its end hold
// -infinity, whose exponential is 0.
template <int G_, int R_, int V_>
struct RowRegs {
    static constexpr int G = G_, R = R_, V = V_;
    // threads of a one-block launch: 1024, or the 512 that leave 256 registers
    // each for the longest rows (128 spill)
    static constexpr int kOneBlock = R * V <= 16 ? kOneBlockThreads : kOneBlockThreads / 2;
    float v[R * V];

    __device__ __forceinline__ static int column(int lane, int i) { return (i * G + lane) * V; }

    __device__ __forceinline__ void load(const float* row, int cols, int lane) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int c = column(lane, i);
            if constexpr (V == 4) {
                const floatx4 q = *reinterpret_cast<const floatx4*>(row + min(c, cols - 4));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * i + e] = q[e];
            } else {
                v[i] = row[min(c, cols - 1)];
            }
        }
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int e = 0; e < V; ++e)
                v[V * i + e] = column(lane, i) < cols ? v[V * i + e] : -INFINITY;
    }

    __device__ __forceinline__ float row_max() const {
        float m = v[0];
#pragma unroll
        for (int i = 1; i < R * V; ++i) m = fmaxf(m, v[i]);
        return group_max<G>(m);
    }

    // v = expf(v - m); returns the row's sum.
    __device__ __forceinline__ float exp_sum(float m) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < R * V; ++i) {
            v[i] = expf(v[i] - m);
            s += v[i];
        }
        return group_sum<G>(s);
    }

    __device__ __forceinline__ void store(float* row, int cols, int lane) const {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int c = column(lane, i);
            if (c >= cols) continue;
            if constexpr (V == 4) {
                *reinterpret_cast<floatx4*>(row + c) =
                    floatx4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
            } else {
                row[c] = v[i];
            }
        }
    }
};

// out[r, :] = exp(x - max) / sum(exp(x - max)).  (Here and below outputs may
// lie over the inputs of the same place, so neither is __restrict__.)
template <class Row>
__global__ void __launch_bounds__(kRowThreads)
softmax_kernel(const float* in, float* out, int64_t rows, int cols) {
    const int lane = threadIdx.x % Row::G;
    const int64_t r = blockIdx.x * (int64_t)(kRowThreads / Row::G) + threadIdx.x / Row::G;
    const int64_t rc = r < rows ? r : rows - 1;  // a group past the end repeats the last row
    Row t;
    t.load(in + rc * cols, cols, lane);
    const float s = t.exp_sum(t.row_max());
#pragma unroll
    for (int i = 0; i < Row::R * Row::V; ++i) t.v[i] /= s;
    if (r < rows) t.store(out + rc * cols, cols, lane);
}

// A row's share of the mean loss, (log(sum exp(z - max)) + max - z_label) /
// batch (0 where the label is no class), and with grad_row its gradient
// (softmax(z) - onehot) / batch.
template <class Row>
__device__ __forceinline__ float xent_row(const float* z, int64_t label, int classes,
                                          float inv_b, int lane, float* grad_row) {
    const bool valid = label >= 0 && label < classes;
    Row t;
    t.load(z, classes, lane);
    const float zl = z[valid ? label : 0];
    const float mx = t.row_max();
    const float s = t.exp_sum(mx);
    if (grad_row) {
        const float inv_s = 1.0f / s;
        // the label's place among this lane's columns, which are compile-time
        // offsets from its first (negative: not here)
        const int at = valid ? (int)label - Row::column(lane, 0) : -1;
#pragma unroll
        for (int i = 0; i < Row::R; ++i)
#pragma unroll
            for (int e = 0; e < Row::V; ++e) {
                float pc = t.v[Row::V * i + e] * inv_s;
                if (at == Row::column(0, i) + e) pc -= 1.0f;
                t.v[Row::V * i + e] = pc * inv_b;
            }
        t.store(grad_row, classes, lane);
    }
    return valid ? (logf(s) + mx - zl) * inv_b : 0.0f;
}

// Cross-entropy over blocks of rows.  Each block adds its rows' loss shares
// and stores the sum at part[block] (part may be null).  The gradients of the
// first `reserved` rows are left out: with many blocks the partial sums lie
// there until xent_finish_kernel has added them, so the call needs no scratch
// memory.
template <class Row>
__global__ void __launch_bounds__(Row::kOneBlock)
xent_kernel(const float* logits, const int64_t* __restrict__ labels, float* part, float* grad,
            int64_t batch, int classes, int64_t reserved) {
    const int lane = threadIdx.x % Row::G;
    const int per_block = blockDim.x / Row::G;
    const float inv_b = 1.0f / (float)batch;
    float lsum = 0.0f;
    int turn = 0;  // the group's lanes take its rows' shares in turn, for short sums
    for (int64_t r0 = blockIdx.x * (int64_t)per_block; r0 < batch;
         r0 += (int64_t)gridDim.x * per_block, turn = (turn + 1) % Row::G) {
        const int64_t r = r0 + threadIdx.x / Row::G;
        const bool live = r < batch;
        const int64_t rc = live ? r : batch - 1;
        float* g = grad && live && r >= reserved ? grad + rc * classes : nullptr;
        const float share =
            xent_row<Row>(logits + rc * classes, labels[rc], classes, inv_b, lane, g);
        if (live && lane == turn) lsum += share;
    }
    if (!part) return;
    const float s = block_sum(lsum);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// One block: loss = the sum of the `nparts` partial sums at the start of grad,
// then the gradients of the `reserved` rows that they lie in.
template <class Row>
__global__ void __launch_bounds__(Row::kOneBlock)
xent_finish_kernel(const float* logits, const int64_t* __restrict__ labels, float* loss,
                   float* grad, int64_t batch, int classes, int nparts, int64_t reserved) {
    const float lsum = thread_partials<Row::kOneBlock>(grad, nparts);
    // (block_sum's barrier comes after every thread's loads of the partial sums)
    const float s = block_sum(lsum);
    if (threadIdx.x == 0) loss[0] = s;
    const int lane = threadIdx.x % Row::G;
    constexpr int kPerBlock = Row::kOneBlock / Row::G;
    const float inv_b = 1.0f / (float)batch;
    for (int64_t r0 = 0; r0 < reserved; r0 += kPerBlock) {
        const int64_t r = r0 + threadIdx.x / Row::G;
        const int64_t rc = r < reserved ? r : reserved - 1;
        (void)xent_row<Row>(logits + rc * classes, labels[rc], classes, inv_b, lane,
                            r < reserved ? grad + rc * classes : nullptr);
    }
}

// Rows too long for registers: a block of 1024 threads per row, which passes
// over the row three times (maximum, sum, output); the later passes find it
// in the L2.  Softmax takes 256 threads per row where there are rows enough to
// fill the CUs with such blocks: 8192 x 2049 65.5 us with 1024, 41.5 with 256
// (46.7 with a wave per row), 20000 x 4096 317 and 275; fewer or longer rows
// need the more threads (2000 x 32000 205 and 218, 256 x 8192 9.4 and 17).
__device__ __forceinline__ float wide_reduce(float x, bool is_max) {
    __shared__ float wred[kOneBlockThreads / kWaveLanes];
    x = is_max ? group_max<kWaveLanes>(x) : group_sum<kWaveLanes>(x);
    __syncthreads();  // the previous reduction's reads are done
    if ((threadIdx.x & (kWaveLanes - 1)) == 0) wred[threadIdx.x / kWaveLanes] = x;
    __syncthreads();
    float s = wred[0];
    for (unsigned w = 1; w < blockDim.x / kWaveLanes; ++w) {
        s = is_max ? fmaxf(s, wred[w]) : s + wred[w];
    }
    return s;
}

__device__ __forceinline__ void wide_max_sum(const float* z, int64_t cols, float& mx, float& s) {
    float m = -INFINITY;
    for (int64_t c = threadIdx.x; c < cols; c += blockDim.x) m = fmaxf(m, z[c]);
    mx = wide_reduce(m, true);
    float e = 0.0f;
    for (int64_t c = threadIdx.x; c < cols; c += blockDim.x) e += expf(z[c] - mx);
    s = wide_reduce(e, false);
}

__global__ void __launch_bounds__(kOneBlockThreads)
softmax_wide_kernel(const float* in, float* out, int64_t rows, int64_t cols) {
    for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
        const float* x = in + r * cols;
        float mx, s;
        wide_max_sum(x, cols, mx, s);
        for (int64_t c = threadIdx.x; c < cols; c += blockDim.x) {
            out[r * cols + c] = expf(x[c] - mx) / s;
        }
    }
}

__device__ __forceinline__ float xent_wide_row(const float* z, int64_t label, int64_t classes,
                                               float inv_b, float* grad_row) {
    const bool valid = label >= 0 && label < classes;
    const float zl = z[valid ? label : 0];
    float mx, s;
    wide_max_sum(z, classes, mx, s);
    if (grad_row) {
        const float inv_s = 1.0f / s;
        for (int64_t c = threadIdx.x; c < classes; c += blockDim.x) {
            float pc = expf(z[c] - mx) * inv_s;
            if (valid && c == label) pc -= 1.0f;
            grad_row[c] = pc * inv_b;
        }
    }
    return valid ? (logf(s) + mx - zl) * inv_b : 0.0f;
}

// As xent_kernel: part[block] = the loss shares of its rows, in row order.
__global__ void __launch_bounds__(kOneBlockThreads)
xent_wide_kernel(const float* logits, const int64_t* __restrict__ labels, float* part,
                 float* grad, int64_t batch, int64_t classes, int64_t reserved) {
    const float inv_b = 1.0f / (float)batch;
    float lsum = 0.0f;
    float lost = 0.0f;  // what the additions to lsum rounded away (Kahan's summation)
    for (int64_t r = blockIdx.x; r < batch; r += gridDim.x) {
        const float share = xent_wide_row(logits + r * classes, labels[r], classes, inv_b,
                                          grad && r >= reserved ? grad + r * classes : nullptr);
        const float y = share - lost;
        const float t = lsum + y;
        lost = fabsf(t) < INFINITY ? (t - lsum) - y : 0.0f;
        lsum = t;
    }
    if (part && threadIdx.x == 0) part[blockIdx.x] = lsum;
}

// As xent_finish_kernel; the partial sums all lie in row 0 (the host keeps
// their number below `classes`).
__global__ void __launch_bounds__(kOneBlockThreads)
xent_wide_finish_kernel(const float* logits, const int64_t* __restrict__ labels,
                        float* loss, float* grad, int64_t batch, int64_t classes,
                        int nparts) {
    const float s = block_sum(thread_partials<kOneBlockThreads>(grad, nparts));
    if (threadIdx.x == 0) loss[0] = s;
    (void)xent_wide_row(logits, labels[0], classes, 1.0f / (float)batch, grad);
}

constexpr int64_t kMaxRegCols = 2048;

inline bool rows_vec4(const void* a, const void* b, int64_t cols) {
    return cols % 4 == 0 &&
           ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15u) == 0;
}

// Calls f with the RowRegs that holds rows of `cols` <= kMaxRegCols columns:
// the fewest lanes that keep a row at no more than 4 values per lane up to 64
// columns (so a wave works on 16 or 4 rows at once; on 64 rows of a single
// column: 1000 x 1, loss and gradient, 4.8 us with four lanes per row, 2.6 with
// one), a whole wave above, with 16-byte accesses where every row starts on a
// 16-byte boundary.
template <class F>
hipError_t with_row_regs(int64_t cols, bool vec4, F&& f) {
    if (cols == 1) return f(RowRegs<1, 1, 1>{});
    if (cols <= 4) return f(RowRegs<4, 1, 1>{});
    if (cols <= 16) return f(RowRegs<4, 4, 1>{});
    if (cols <= 64) return f(RowRegs<16, 4, 1>{});
    if (vec4) {
        if (cols <= 256) return f(RowRegs<64, 1, 4>{});
        if (cols <= 512) return f(RowRegs<64, 2, 4>{});
        if (cols <= 1024) return f(RowRegs<64, 4, 4>{});
        return f(RowRegs<64, 8, 4>{});
    }
    if (cols <= 128) return f(RowRegs<64, 2, 1>{});
    if (cols <= 256) return f(RowRegs<64, 4, 1>{});
    if (cols <= 512) return f(RowRegs<64, 8, 1>{});
    if (cols <= 1024) return f(RowRegs<64, 16, 1>{});
    return f(RowRegs<64, 32, 1>{});
}

}  // namespace

hipError_t launch_softmax(const float* in, float* out, int64_t rows, int64_t cols,
                          hipStream_t stream) {
    if (rows == 0 || cols == 0) return hipSuccess;
    if (cols > kMaxRegCols) {
        const unsigned blocks = (unsigned)std::min<int64_t>(rows, 1 << 20);
        const int threads = rows >= 4096 && cols <= 16384 ? kRowThreads : kOneBlockThreads;
        hipLaunchKernelGGL(softmax_wide_kernel, dim3(blocks), dim3(threads), 0, stream, in, out,
                           rows, cols);
        return hipGetLastError();
    }
    return with_row_regs(cols, rows_vec4(in, out, cols), [&](auto row) {
        using Row = decltype(row);
        constexpr int kPerBlock = kRowThreads / Row::G;
        hipLaunchKernelGGL((softmax_kernel<Row>), dim3((unsigned)((rows + kPerBlock - 1) / kPerBlock)),
                           dim3(kRowThreads), 0, stream, in, out, rows, (int)cols);
        return hipGetLastError();
    });
}

int64_t xent_parts(int64_t batch, int64_t classes) {
    if (classes > kMaxRegCols) return std::min<int64_t>(batch, kMaxRowBlocks);
    int64_t blocks = 0;
    (void)with_row_regs(classes, false, [&](auto row) {
        constexpr int kPerBlock = kRowThreads / decltype(row)::G;
        blocks = std::min<int64_t>((batch + kPerBlock - 1) / kPerBlock, kMaxRowBlocks);
        return hipSuccess;
    });
    return blocks;
}

hipError_t launch_xent_parts(const float* logits, const int64_t* labels, float* part, float* grad,
                             int64_t batch, int64_t classes, hipStream_t stream) {
    const dim3 grid((unsigned)xent_parts(batch, classes));
    if (classes > kMaxRegCols) {
        hipLaunchKernelGGL(xent_wide_kernel, grid, dim3(kOneBlockThreads), 0, stream, logits,
                           labels, part, grad, batch, classes, (int64_t)0);
        return hipGetLastError();
    }
    return with_row_regs(classes, rows_vec4(logits, grad, classes), [&](auto row) {
        using Row = decltype(row);
        hipLaunchKernelGGL((xent_kernel<Row>), grid, dim3(kRowThreads), 0, stream, logits, labels,
                           part, grad, batch, (int)classes, (int64_t)0);
        return hipGetLastError();
    });
}

// Many blocks and a second launch that adds their loss sums, unless one block
// takes the batch in few rounds of its 1024 threads: three of up to 4 columns
// per thread (about 1 us each: 513 x 10 in three rounds 4.5 us against 4.8 us
// for two launches, 1024 x 10 in four 5.8 against 4.8), one of longer rows
// (16 x 1000 4.4 us; 33 x 1000 in three rounds 9.3 us against 6.3), or nothing can hold the sums between the launches:
// no gradient buffer (loss only), or one that overlaps the logits.
// 4096 x 1000, loss and gradient: 10.3 ms with one thread per row on one
// block, 11.3 us now (33 MB: 2.9 TB/s; the gradient launch alone 4.4 TB/s).
hipError_t launch_softmax_xent(const float* logits, const int64_t* labels, float* loss,
                               float* grad, int64_t batch, int64_t classes, hipStream_t stream) {
    const int64_t n = batch * classes;
    const bool overlap = grad && grad < logits + n && logits < grad + n;
    const bool one_only = loss && (!grad || overlap);
    if (classes > kMaxRegCols) {
        const int blocks = one_only ? 1 : (int)std::min({batch, classes, (int64_t)kMaxRowBlocks});
        const bool two = loss && blocks > 1;
        hipLaunchKernelGGL(xent_wide_kernel, dim3(blocks), dim3(kOneBlockThreads), 0, stream,
                           logits, labels, two ? grad : loss, grad, batch, classes, two ? 1 : 0);
        if (two) {
            hipLaunchKernelGGL(xent_wide_finish_kernel, dim3(1), dim3(kOneBlockThreads), 0, stream,
                               logits, labels, loss, grad, batch, classes, blocks);
        }
        return hipGetLastError();
    }
    const bool vec4 = rows_vec4(logits, grad, classes);
    return with_row_regs(classes, vec4, [&](auto row) {
        using Row = decltype(row);
        constexpr int kPerBlock = kRowThreads / Row::G;
        constexpr int kPerOne = Row::kOneBlock / Row::G;
        constexpr int kRounds = Row::R * Row::V <= 4 ? 3 : 1;
        const bool one = one_only || (loss && batch <= kRounds * kPerOne);
        // (rows of a few columns: fewer sums, as many rows hold few of them)
        constexpr int kMost = Row::G == kWaveLanes ? kMaxRowBlocks : kMaxRowBlocks / 4;
        const int blocks =
            one ? 1 : (int)std::min<int64_t>((batch + kPerBlock - 1) / kPerBlock, kMost);
        const bool two = loss && blocks > 1;
        const int64_t reserved = two ? (blocks + classes - 1) / classes : 0;
        hipLaunchKernelGGL((xent_kernel<Row>), dim3(blocks),
                           dim3(one ? Row::kOneBlock : kRowThreads), 0, stream, logits, labels,
                           two ? grad : loss, grad, batch, (int)classes, reserved);
        if (two) {
            hipLaunchKernelGGL((xent_finish_kernel<Row>), dim3(1), dim3(Row::kOneBlock), 0,
                               stream, logits, labels, loss, grad, batch, (int)classes, blocks,
                               reserved);
        }
        return hipGetLastError();
    });
}

}  // namespace fdl
