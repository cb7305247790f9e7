// Two small decode-step kernels next to the three operators: the SwiGLU elementwise product
// silu(a) * b (model.py:134 evaluates it with two torch kernels) and the greedy argmax over the
// logits row (model.py:371).  In a graph-replayed decode step both are dispatch-bound; one
// launch each instead of two resp. a 40 us single-workgroup library reduction.
#include <algorithm>

#include "l3_device.hpp"
#include "l3_host.hpp"

namespace l3 {

namespace {

constexpr int kMiscThreads = 256;
constexpr int kArgmaxWide = 2048;   // workgroups of the argmax from which on they take four times the logits

// y = bf16( bf16(silu(a)) * b ) with silu_rounded of l3_device.hpp.

// blockIdx.y walks over the rows (no index division in the lanes); rows of a and b may be strided
// (the two halves of one fused gate|up projection), y is dense.
__global__ void __launch_bounds__(kMiscThreads)
silu_mul_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, uint16_t* __restrict__ y,
                int64_t rows, int64_t vec_per_row, int64_t a_row_stride, int64_t b_row_stride) {
    const int64_t col = int64_t(blockIdx.x) * kMiscThreads + threadIdx.x;
    if (col >= vec_per_row) return;
    for (int64_t row = blockIdx.y; row < rows; row += gridDim.y) {
        float fa[8], fb[8];
        unpack8(load16(a + row * a_row_stride + col * 8), fa);
        unpack8(load16(b + row * b_row_stride + col * 8), fb);
        uint4 o;
        o.x = pack_bf16x2(silu_rounded(fa[0]) * fb[0], silu_rounded(fa[1]) * fb[1]);
        o.y = pack_bf16x2(silu_rounded(fa[2]) * fb[2], silu_rounded(fa[3]) * fb[3]);
        o.z = pack_bf16x2(silu_rounded(fa[4]) * fb[4], silu_rounded(fa[5]) * fb[5]);
        o.w = pack_bf16x2(silu_rounded(fa[6]) * fb[6], silu_rounded(fa[7]) * fb[7]);
        store16(y + (row * vec_per_row + col) * 8, o);
    }
}

__global__ void __launch_bounds__(kMiscThreads)
silu_mul_scalar_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, uint16_t* __restrict__ y,
                       int64_t n) {
    const int64_t i = int64_t(blockIdx.x) * kMiscThreads + threadIdx.x;
    if (i >= n) return;
    y[i] = uint16_t(f32_to_bf16_bits(silu_rounded(bf16_to_f32(a[i])) * bf16_to_f32(b[i])));
}

// Order of bf16 logits as 16-bit whole numbers: the first maximum wins, as torch.argmax documents (so -0 counts
// as 0), and a NaN ranks above every number (the first NaN wins), which is how torch.argmax treats it: a
// numerical blow-up shows up in the token stream the same way on both paths.  No logit has order 0.
__device__ __forceinline__ uint32_t logit_order(uint32_t bits) {
    const uint32_t up = (bits & 0x8000u) ? ~bits & 0xffffu : bits | 0x8000u;
    return (bits & 0x7fffu) > 0x7f80u ? 0xffffu : bits == 0x8000u ? 0x8000u : up;
}

// Stage 1: a workgroup scans U * 2048 logits of one row and writes its best one as order << 32 | ~index; stage 2
// takes the largest such word of a row.  Bound by latency: order and place within the workgroup share a 32-bit
// word, so that eight logits of a 16-byte load cost one maximum each and a lane exchange moves one register, and all
// loads of a thread are in flight together.  Both stages, 1 / 16 / 64 rows of 128256 logits, recorded: 6.6 / 8.2 /
// 15.0 us with 2-byte loads and (value, index) pairs, 3.7 / 4.8 / 7.3 us now.
template <int U>
__global__ void __launch_bounds__(kMiscThreads)
argmax_partial_kernel(const uint16_t* __restrict__ logits, int64_t row_stride, int V, bool vec, uint64_t* __restrict__ part) {
    constexpr int CHUNK = U * kArgmaxChunk;
    static_assert(kArgmaxChunk == kMiscThreads * 8 && CHUNK <= 65536, "a 16-byte load per thread; places in 16 bits");
    const int c0 = int(blockIdx.x) * CHUNK;
    const int n = min(V - c0, CHUNK);
    const uint16_t* r = logits + blockIdx.y * row_stride + c0;
    uint32_t best = 0;
    auto take = [&](uint32_t bits, int place) __attribute__((always_inline)) {
        best = max(best, logit_order(bits) << 16 | (0xffffu - uint32_t(place)));
    };
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = (u * kMiscThreads + int(threadIdx.x)) * 8;
        if (vec && i + 8 <= n) v[u] = load16(r + i);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int i = (u * kMiscThreads + int(threadIdx.x)) * 8;
        if (vec && i + 8 <= n) {
            const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                take(w[j] & 0xffffu, i + 2 * j);
                take(w[j] >> 16, i + 2 * j + 1);
            }
        } else {
            for (int j = i; j < min(i + 8, n); ++j) take(r[j], j);
        }
    }
#pragma unroll
    for (int off = 1; off < kWaveSize; off <<= 1) best = max(best, uint32_t(__shfl_xor(int(best), off, kWaveSize)));
    __shared__ uint32_t s_best[kMiscThreads / kWaveSize];
    if ((threadIdx.x & (kWaveSize - 1)) == 0) s_best[threadIdx.x / kWaveSize] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < kMiscThreads / kWaveSize; ++w) best = max(best, s_best[w]);
        part[int64_t(blockIdx.y) * gridDim.x + blockIdx.x] = uint64_t(best >> 16) << 32 | ~uint32_t(c0 + int(0xffffu - (best & 0xffffu)));
    }
}

__device__ __forceinline__ uint64_t best_of_parts(const uint64_t* part, int nparts, int lane) {
    uint64_t best = 0;
    for (int i = lane; i < nparts; i += kWaveSize) best = max(best, part[i]);
    return best;
}
__device__ __forceinline__ uint64_t best_of_wave(uint64_t best) {
#pragma unroll
    for (int off = 1; off < kWaveSize; off <<= 1) {
        best = max(best, uint64_t(__shfl_xor(static_cast<unsigned long long>(best), off, kWaveSize)));
    }
    return best;
}
__device__ __forceinline__ int64_t best_index(uint64_t best) { return int64_t(~uint32_t(best)); }

__global__ void __launch_bounds__(kWaveSize)
argmax_final_kernel(const uint64_t* __restrict__ part, int nparts, int64_t* __restrict__ out) {
    const uint64_t best = best_of_wave(best_of_parts(part + int64_t(blockIdx.x) * nparts, nparts, int(threadIdx.x)));
    if (threadIdx.x == 0) out[blockIdx.x] = best_index(best);
}

// Second argmax stage fused with the bookkeeping generate() does per greedy token
// (model.py:371-378): with next = pos + 1 (clamped to the last column),
//   nxt = text_mask[b, next] ? tokens[b, next] : argmax(logits[b])     (a prompt token is kept)
//   tokens[b, next] = nxt;  tok[b] = nxt (the token fed to the next step)
//   eos[b] |= !text_mask[b, next] && nxt is a stop token
// and pos += 1, kv_len += 1.  One workgroup handles all rows (a wavefront per four rows in turn).  In a
// graph-replayed decode step this stands for the second argmax stage plus about a dozen tiny elementwise
// launches.  Bound by its chain of dependent accesses, so nothing waits that need not: the position, the stop tokens and
// the parts are read together, the counters move on as soon as everybody has the position, and only the tokens of that
// position are read behind it.  With the first stage, 1 / 64 rows: 10.5 / 21.4 us with the counters behind all stores
// and the stop tokens read one after the other, 5.6 / 11.2 us now.
constexpr int kGreedyThreads = 1024;
constexpr int kGreedyRowsPerPass = 4;   // rows a wavefront takes per pass, loads of all of them in flight together
__global__ void __launch_bounds__(kGreedyThreads)
greedy_step_kernel(const uint64_t* __restrict__ part, int nparts, int rows,
                   int64_t* __restrict__ tokens, const uint8_t* __restrict__ text_mask, int64_t total_len,
                   int64_t* __restrict__ tok, int* __restrict__ pos, int* __restrict__ kv_len,
                   uint8_t* __restrict__ eos, const int64_t* __restrict__ stop, int n_stop) {
    constexpr int NWAVES = kGreedyThreads / kWaveSize;
    constexpr int RP = kGreedyRowsPerPass;
    const int lane = threadIdx.x & (kWaveSize - 1);
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWaveSize);
    const int p0 = *pos, len0 = *kv_len;
    const int64_t stop0 = lane < n_stop ? stop[lane] : 0;
    uint64_t best[RP];
    auto read_parts = [&](int base) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < RP; ++j) best[j] = best_of_parts(part + int64_t(min(base + j, rows - 1)) * nparts, nparts, lane);
    };
    if (wave * RP < rows) read_parts(wave * RP);
    __syncthreads();   // everybody has the position
    if (threadIdx.x == 0) {
        *pos = p0 + 1;
        *kv_len = len0 + 1;
    }
    const int64_t next = min(int64_t(p0) + 1, total_len - 1);
    for (int base = wave * RP; base < rows; base += NWAVES * RP) {
        if (base != wave * RP) read_parts(base);
        bool keep[RP];
        int64_t prompt_tok[RP];
#pragma unroll
        for (int j = 0; j < RP; ++j) {
            const int row = min(base + j, rows - 1);
            keep[j] = text_mask[row * total_len + next] != 0;
            prompt_tok[j] = tokens[row * total_len + next];
        }
#pragma unroll
        for (int j = 0; j < RP; ++j) {
            const int row = base + j;
            int64_t nxt = best_index(best_of_wave(best[j]));
            if (keep[j]) nxt = prompt_tok[j];
            bool is_stop = lane < n_stop && stop0 == nxt;
            for (int i = lane + kWaveSize; i < n_stop; i += kWaveSize) is_stop |= stop[i] == nxt;
            is_stop = __builtin_amdgcn_ballot_w64(is_stop) != 0;
            if (lane == 0 && row < rows) {
                tokens[row * total_len + next] = nxt;
                tok[row] = nxt;
                if (!keep[j] && is_stop) eos[row] = 1;
            }
        }
    }
}

// Logits of all rows in one grid: 2048 per workgroup, or 8192 where that still fills the device twice (fewer parts for
// the second stage to read).
int launch_argmax_partial(const uint16_t* logits, int64_t row_stride, int rows, int V, uint64_t* part, int* parts, hipStream_t stream) {
    const bool vec = reinterpret_cast<uintptr_t>(logits) % 16 == 0 && (rows == 1 || row_stride % 8 == 0);
    *parts = argmax_parts(V);
    if (int64_t(rows) * *parts < kArgmaxWide) {
        return enqueue(argmax_partial_kernel<1>, dim3(unsigned(*parts), unsigned(rows)), dim3(kMiscThreads), 0, stream, logits,
                       row_stride, V, vec, part);
    }
    *parts = (*parts + 3) / 4;
    return enqueue(argmax_partial_kernel<4>, dim3(unsigned(*parts), unsigned(rows)), dim3(kMiscThreads), 0, stream, logits,
                   row_stride, V, vec, part);
}

}  // namespace

int launch_greedy_step(const uint16_t* logits, int64_t row_stride, int rows, int V, uint64_t* part, int64_t* tokens,
                       const uint8_t* text_mask, int64_t total_len, int64_t* tok, int* pos, int* kv_len, uint8_t* eos,
                       const int64_t* stop, int n_stop, hipStream_t stream) {
    int parts;
    if (const int rc = launch_argmax_partial(logits, row_stride, rows, V, part, &parts, stream); rc != 0) return rc;
    return enqueue(greedy_step_kernel, dim3(1), dim3(kGreedyThreads), 0, stream, part, parts, rows, tokens, text_mask,
                   total_len, tok, pos, kv_len, eos, stop, n_stop);
}

int launch_silu_mul_rows(const uint16_t* a, const uint16_t* b, uint16_t* y, int64_t rows, int64_t cols,
                         int64_t a_row_stride, int64_t b_row_stride, hipStream_t stream) {
    const int64_t vpr = cols / 8;
    const dim3 grid(unsigned((vpr + kMiscThreads - 1) / kMiscThreads), unsigned(std::min<int64_t>(rows, 65535)));
    return enqueue(silu_mul_kernel, grid, dim3(kMiscThreads), 0, stream, a, b, y, rows, vpr, a_row_stride,
                   b_row_stride);
}

int launch_silu_mul(const uint16_t* a, const uint16_t* b, uint16_t* y, int64_t n, bool vec_ok, hipStream_t stream) {
    if (vec_ok) {
        const int64_t nvec = n / 8;
        return enqueue(silu_mul_kernel, dim3(unsigned((nvec + kMiscThreads - 1) / kMiscThreads)),
                       dim3(kMiscThreads), 0, stream, a, b, y, int64_t(1), nvec, int64_t(0), int64_t(0));
    } else {
        return enqueue(silu_mul_scalar_kernel, dim3(unsigned((n + kMiscThreads - 1) / kMiscThreads)),
                       dim3(kMiscThreads), 0, stream, a, b, y, n);
    }
}

int argmax_parts(int V) { return (V + kArgmaxChunk - 1) / kArgmaxChunk; }

int launch_argmax(const uint16_t* logits, int64_t row_stride, int rows, int V, uint64_t* part, int64_t* out, hipStream_t stream) {
    int parts;
    if (const int rc = launch_argmax_partial(logits, row_stride, rows, V, part, &parts, stream); rc != 0) return rc;
    return enqueue(argmax_final_kernel, dim3(unsigned(rows)), dim3(kWaveSize), 0, stream, part, parts, out);
}

}  // namespace l3
