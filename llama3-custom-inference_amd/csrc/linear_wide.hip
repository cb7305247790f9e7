// y[M, N] = x[M, K] . W[N, K]^T for up to 64 activation rows: the nn.Linear calls of model.py:95,121,134,225
// at decode batch sizes where the activations no longer fit one matrix-instruction column block.
//
// Bound by the stream over the weight matrix; what it takes to reach it (weights of 16 layers in turn, graph
// replays, 64 rows):
//   * Both operands go from memory straight into LDS (buffer_load_dwordx4 ... lds), 256 contiguous bytes of a
//     row per 16 lanes, in a ring of ST stages of 128 k each.  Loading the activations into operand registers
//     instead (64-byte pieces of 16 rows per instruction, half of the instructions for data that every
//     workgroup re-reads) kept the vector memory pipe busier than the weights did: 28 us for the gate|up
//     pair 2 x 8192 x 2048, against 16 us through LDS.
//   * One barrier per 128 k.  The wait before it counts the loads of the newer stages, which stay in flight; the
//     loads are issued by inline assembly, because the compiler otherwise waits for all of them before it
//     reads LDS at the head of the loop.
//   * The workgroups start at different places of their k range: rows lie K * 2 bytes apart, usually a multiple
//     of 4096, so workgroups that walk in step would ask the same memory channels (gate|up 16.0 -> 14.3 us).
//   * Rows are not padded in LDS: the 16-byte chunk c of row r sits at position c ^ (r & 15), which spreads the
//     rows of an operand read over all banks.
// Measured against what ran before (a library GEMM plus the SwiGLU product: 21.2 us): gate|up 14.4 us; down
// projection 2048 x 8192 in 8 splits 11.8 -> 9.9 us; out projection 2048 x 2048 5.5 -> 5.0 us; qkv 3072 x 2048
// 7.0 -> 6.6 us; vocabulary projection 128256 x 2048 107 (library GEMM) -> 95 us.
#include <algorithm>

#include "lds_loads.hpp"

namespace l3 {

namespace {

constexpr int kWideWaves = 8;
constexpr int kWideChunk = 128;                  // k per stage
constexpr int kWideRowBytes = kWideChunk * 2;    // of one row in a stage

struct WideParams {
    const uint16_t* x;    // (M, K)
    const uint16_t* w0;   // (N, K)
    const uint16_t* w1;   // second matrix of the SwiGLU form
    const uint16_t* res;  // (M, N) residual added to y, y's row stride (else null)
    uint16_t* y;          // (M, N) bf16, or ...
    float* part;          // ... (splits, M, N) partial products
    int M, N, K;
    uint32_t x_pitch, w_pitch;   // bytes from a row to the next
    int64_t y_stride;
    int row_groups, chunks_per_split;
    QkvTarget qkv;
};

enum class WideOut { kPartials, kSwiglu, kRows, kQkv };

// Features n .. n + 3 (n % 4 == 0) of activation row m of a qkv projection, rounded to bf16: query and key pairs are
// rotated at the device-side position, keys and values go into the cache row of that position (model.py:100-106).
__device__ __forceinline__ void store_qkv(const QkvTarget& t, int m, int n, const f32x4_t& s) {
    const int pos = *t.pos;
    if (pos < 0 || pos >= t.cache_len || pos >= t.table_rows) return;   // never write outside the cache
    const int slot = n / t.HD, d = n % t.HD;
    uint2 v = make_uint2(pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3]));
    uint16_t* to = t.q_out + (int64_t(m) * t.NH + slot) * t.HD + d;
    if (slot < t.NH + t.KVH) {
        const float4 cs = *reinterpret_cast<const float4*>(t.table + int64_t(pos) * t.HD + d);
        v.x = rotate_pair(v.x, cs.x, cs.y);
        v.y = rotate_pair(v.y, cs.z, cs.w);
        if (slot >= t.NH) to = t.cache_k + m * t.c_sb + pos * t.c_st + (slot - t.NH) * t.HD + d;
    } else {
        to = t.cache_v + m * t.c_sb + pos * t.c_st + (slot - t.NH - t.KVH) * t.HD + d;
    }
    *reinterpret_cast<uint2*>(to) = v;
}

// CB: blocks of 16 activation rows.  RF: blocks of 16 weight rows per wavefront (SwiGLU: half of them of each
// matrix).  The eight wavefronts are WR (weight rows) x WC (activation rows) x WK (k steps of a stage); WK
// of them meet in LDS at the end.  A workgroup is one (row group, k range), or with kQkv one (row group, 16 CB of the
// activation rows).
template <int CB, int RF, int WR, int WC, int WK, int ST, WideOut OUT>
__global__ void __launch_bounds__(kWideWaves * kWaveSize)
linear_wide_kernel(const WideParams p) {
    static_assert(WR * WC * WK == kWideWaves && CB % WC == 0, "wavefronts");
    constexpr bool SWIGLU = OUT == WideOut::kSwiglu;
    constexpr int ROWS = 16 * RF * WR;                      // weight rows a workgroup streams
    constexpr int N_WG = SWIGLU ? ROWS / 2 : ROWS;          // outputs per activation row
    constexpr int CBW = CB / WC, KSW = 4 / WK;              // column blocks and k steps per wavefront
    constexpr int RO = SWIGLU ? RF / 2 : RF;                // blocks of output rows per wavefront
    constexpr int WI = ROWS / 32;                           // weight loads per wavefront and stage (1 KiB: four rows)
    constexpr int XI = (CB * 4 + kWideWaves - 1) / kWideWaves;   // activation loads (with one block some are issued twice)
    constexpr int NI = WI + XI;
    constexpr int WBYTES = ROWS * kWideRowBytes, STAGE = WBYTES + CB * 16 * kWideRowBytes;
    __shared__ __align__(1024) unsigned char s_ring[ST * STAGE];

    const int lane = threadIdx.x & (kWaveSize - 1);
    const int wave = wave_uniform(int(threadIdx.x) / kWaveSize);
    const int fn = lane & 15, fg = lane >> 4;
    const int wr = wave % WR, wc = (wave / WR) % WC, wk = wave / (WR * WC);
    const int group = int(blockIdx.x) % p.row_groups, part = int(blockIdx.x) / p.row_groups;
    const int split = OUT == WideOut::kQkv ? 0 : part, m0 = OUT == WideOut::kQkv ? part * (CB * 16) : 0;
    const int n0 = group * N_WG;
    const int c0 = split * p.chunks_per_split;
    const int n_chunks = min(p.K / kWideChunk, c0 + p.chunks_per_split) - c0;   // (none: the split's products are zeros)

    // loads: lane l of a load covers row l / 16 of its four rows, chunk position l % 16
    const uint32_t ring = lds_address(s_ring);
    // (row groups of four are all inside N or all outside: those outside re-read the last one and are never stored;
    // one resource per load keeps the lane offsets below four row pitches)
    const int ld_row = lane >> 4;
    uint32_t woff[WI], xoff[XI];
    srd_t bw[WI], bx[XI];
#pragma unroll
    for (int j = 0; j < WI; ++j) {
        const int first = (wave * WI + j) * 4;              // of the workgroup's rows; a load is all gate or all up
        const bool up = SWIGLU && first >= N_WG;
        const int row = min(n0 + (up ? first - N_WG : first), p.N - 4);
        bw[j] = make_srd(reinterpret_cast<const char*>(up ? p.w1 : p.w0) + int64_t(row) * p.w_pitch);
        woff[j] = uint32_t(ld_row) * p.w_pitch + uint32_t(((lane & 15) ^ ((first + ld_row) & 15)) * 16);
    }
#pragma unroll
    for (int j = 0; j < XI; ++j) {
        const int first = ((wave * XI + j) % (CB * 4)) * 4;
        const int row = min(m0 + first, p.M - 1);
        bx[j] = make_srd(reinterpret_cast<const char*>(p.x) + int64_t(row) * p.x_pitch);
        xoff[j] = uint32_t(min(ld_row, p.M - 1 - row)) * p.x_pitch + uint32_t(((lane & 15) ^ ((first + ld_row) & 15)) * 16);
    }
    int next = (split == 0 && p.chunks_per_split >= 8) ? (group * 3) % n_chunks : 0;   // splits already start apart
    auto request = [&](int slot) __attribute__((always_inline)) {
        const int koff = (c0 + next) * kWideRowBytes;
        const uint32_t stage = ring + uint32_t(slot * STAGE);
#pragma unroll
        for (int j = 0; j < WI; ++j) {
            load_to_lds<true>(bw[j], stage + (wave * WI + j) * 1024, woff[j], koff);
        }
#pragma unroll
        for (int j = 0; j < XI; ++j) {
            load_to_lds<false>(bx[j], stage + WBYTES + ((wave * XI + j) % (CB * 4)) * 1024, xoff[j], koff);
        }
        if (++next == n_chunks) next = 0;
    };

    f32x4_t acc[RF][CBW];
#pragma unroll
    for (int r = 0; r < RF; ++r) {
#pragma unroll
        for (int c = 0; c < CBW; ++c) acc[r][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    auto multiply = [&](const unsigned char* stage) __attribute__((always_inline)) {
        uint4 a[KSW][RF], b[KSW][CBW];
#pragma unroll
        for (int s = 0; s < KSW; ++s) {
            const int pos = (((wk * KSW + s) * 4 + fg) ^ fn) * 16;
#pragma unroll
            for (int r = 0; r < RF; ++r) {
                const int block = (SWIGLU && r >= RO) ? N_WG / 16 + wr * RO + r - RO : wr * RO + r;
                a[s][r] = *reinterpret_cast<const uint4*>(stage + (block * 16 + fn) * kWideRowBytes + pos);
            }
#pragma unroll
            for (int c = 0; c < CBW; ++c) {
                b[s][c] = *reinterpret_cast<const uint4*>(stage + WBYTES + ((wc * CBW + c) * 16 + fn) * kWideRowBytes + pos);
            }
        }
#pragma unroll
        for (int s = 0; s < KSW; ++s) {
#pragma unroll
            for (int r = 0; r < RF; ++r) {
#pragma unroll
                for (int c = 0; c < CBW; ++c) {
                    acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[s][r]),
                                                                        __builtin_bit_cast(bf16x8_t, b[s][c]), acc[r][c], 0, 0, 0);
                }
            }
        }
    };

#pragma unroll
    for (int d = 0; d < ST - 1; ++d) {
        if (d < n_chunks) request(d);
    }
    for (int t = 0; t < n_chunks; t += ST) {
#pragma unroll
        for (int d = 0; d < ST; ++d) {
            if (t + d < n_chunks) {   // workgroup-uniform
                // this wavefront's part of the stage has landed, then everybody's; the stage that is requested next was
                // last read before this barrier
                if (t + d + ST - 2 < n_chunks) wait_loads<NI*(ST - 2)>(); else wait_loads<0>();
                barrier_after_lds();
                if (t + d + ST - 1 < n_chunks) request((d + ST - 1) % ST);
                multiply(s_ring + d * STAGE);
            }
        }
    }

    // acc[r][c][i]: weight row 16 block + 4 fg + i against activation row 16 (wc CBW + c) + fn
    auto store = [&](int block, int cblock, int l, const f32x4_t& s, const f32x4_t& u) __attribute__((always_inline)) {
        const int m = m0 + cblock * 16 + (l & 15), n = n0 + block * 16 + 4 * (l >> 4);
        if (m >= p.M || n >= p.N) return;
        if constexpr (OUT == WideOut::kPartials) {
            *reinterpret_cast<f32x4_t*>(p.part + (int64_t(split) * p.M + m) * p.N + n) = s;
        } else if constexpr (OUT == WideOut::kQkv) {
            store_qkv(p.qkv, m, n, s);
        } else {
            float o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                o[i] = s[i];
                if constexpr (SWIGLU) {
                    const float g = __uint_as_float(f32_to_bf16_bits(s[i]) << 16);
                    o[i] = silu_rounded(g) * __uint_as_float(f32_to_bf16_bits(u[i]) << 16);
                }
            }
            uint2 v;
            v.x = pack_bf16x2(o[0], o[1]);
            v.y = pack_bf16x2(o[2], o[3]);
            if (p.res) {   // bf16(residual + bf16(product)), as the separate addition would give
                const uint2 r = *reinterpret_cast<const uint2*>(p.res + int64_t(m) * p.y_stride + n);
                v.x = pack_bf16x2(bf16lo_to_f32(r.x) + bf16lo_to_f32(v.x), bf16hi_to_f32(r.x) + bf16hi_to_f32(v.x));
                v.y = pack_bf16x2(bf16lo_to_f32(r.y) + bf16lo_to_f32(v.y), bf16hi_to_f32(r.y) + bf16hi_to_f32(v.y));
            }
            *reinterpret_cast<uint2*>(p.y + int64_t(m) * p.y_stride + n) = v;
        }
    };
    if constexpr (OUT == WideOut::kRows && WK == 1) {
        // Whole 128-byte lines: the tile is turned in LDS and a row's outputs leave 16 bytes per lane, non-temporal
        // (64 rows of the vocabulary projection are 16 MB among half a gigabyte of weights: 8-byte stores straight
        // from the accumulators 109 us, whole lines 108, non-temporal 100, with two workgroups per unit 95).
        static_assert(ROWS % 64 == 0, "whole lines");
        constexpr int CPM = ROWS / 8;   // 16-byte chunks of an activation row's outputs
        static_assert(CB * 16 * ROWS * 2 <= ST * STAGE, "tile");
        constexpr int PIECES = CB * 16 * CPM, NT = kWideWaves * kWaveSize;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < RF; ++r) {
#pragma unroll
            for (int c = 0; c < CBW; ++c) {
                const int m = (wc * CBW + c) * 16 + fn, n = (wr * RF + r) * 16 + 4 * fg;
                uint2 v;
                v.x = pack_bf16x2(acc[r][c][0], acc[r][c][1]);
                v.y = pack_bf16x2(acc[r][c][2], acc[r][c][3]);
                *reinterpret_cast<uint2*>(s_ring + m * (ROWS * 2) + (((n / 8) ^ (m & (CPM - 1))) * 16) + (n & 4) * 2) = v;
            }
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < (PIECES + NT - 1) / NT; ++it) {
            const int idx = int(threadIdx.x) + it * NT;
            if (PIECES % NT != 0 && idx >= PIECES) break;
            const int m = idx / CPM, ch = idx % CPM;
            u32x4_t v = *reinterpret_cast<const u32x4_t*>(s_ring + m * (ROWS * 2) + ((ch ^ (m & (CPM - 1))) * 16));
            if (m < p.M && n0 + ch * 8 < p.N) {
                if (p.res) {
                    const u32x4_t r = *reinterpret_cast<const u32x4_t*>(p.res + int64_t(m) * p.y_stride + n0 + ch * 8);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        v[i] = pack_bf16x2(bf16lo_to_f32(r[i]) + bf16lo_to_f32(v[i]), bf16hi_to_f32(r[i]) + bf16hi_to_f32(v[i]));
                    }
                }
                __builtin_nontemporal_store(v, reinterpret_cast<u32x4_t*>(p.y + int64_t(m) * p.y_stride + n0 + ch * 8));
            }
        }
    } else if constexpr (WK == 1) {
#pragma unroll
        for (int r = 0; r < RO; ++r) {
#pragma unroll
            for (int c = 0; c < CBW; ++c) store(wr * RO + r, wc * CBW + c, lane, acc[r][c], acc[SWIGLU ? r + RO : r][c]);
        }
    } else {
        static_assert(kWideWaves * RF * CBW * 1024 <= ST * STAGE, "the sums meet in the ring");
        __syncthreads();
        auto slot = [&](int w, int r, int c) { return reinterpret_cast<float*>(s_ring) + ((w * RF + r) * CBW + c) * 256; };
#pragma unroll
        for (int r = 0; r < RF; ++r) {
#pragma unroll
            for (int c = 0; c < CBW; ++c) *reinterpret_cast<f32x4_t*>(slot(wave, r, c) + lane * 4) = acc[r][c];
        }
        __syncthreads();
        constexpr int BLOCKS = WR * WC * RO * CBW;   // output blocks of the workgroup, dealt to the wavefronts
#pragma unroll
        for (int it = 0; it < (BLOCKS + kWideWaves - 1) / kWideWaves; ++it) {
            const int f = wave + it * kWideWaves;
            if (f < BLOCKS) {   // wave-uniform
                const int w = f / (RO * CBW), r = f % (RO * CBW) / CBW, c = f % CBW;
                f32x4_t s = {0.f, 0.f, 0.f, 0.f}, u = s;
#pragma unroll
                for (int k = 0; k < WK; ++k) {
                    s += *reinterpret_cast<const f32x4_t*>(slot(k * WR * WC + w, r, c) + lane * 4);
                    if constexpr (SWIGLU) u += *reinterpret_cast<const f32x4_t*>(slot(k * WR * WC + w, r + RO, c) + lane * 4);
                }
                store((w % WR) * RO + r, (w / WR) * CBW + c, lane, s, u);
            }
        }
    }
}

template <int CB, int RF, int WR, int WC, int WK, int ST, WideOut OUT>
int launch_variant(WideParams p, int ksplit, hipStream_t stream) {   // (kQkv: groups of activation rows)
    constexpr int N_WG = 16 * RF * WR / (OUT == WideOut::kSwiglu ? 2 : 1);
    p.row_groups = (p.N + N_WG - 1) / N_WG;
    p.chunks_per_split = OUT == WideOut::kQkv ? p.K / kWideChunk : (p.K / kWideChunk + ksplit - 1) / ksplit;
    return enqueue(linear_wide_kernel<CB, RF, WR, WC, WK, ST, OUT>, dim3(unsigned(p.row_groups) * unsigned(ksplit)),
                   dim3(kWideWaves * kWaveSize), 0, stream, p);
}

// Blocks of 16 activation rows -> the kernel for them.
template <int RF, int ST, WideOut OUT>
int launch_by_rows(const WideParams& p, int ksplit, hipStream_t stream) {
    if (p.M <= 16) return launch_variant<1, RF, 2, 1, 4, ST, OUT>(p, ksplit, stream);
    if (p.M <= 32) return launch_variant<2, RF, 2, 1, 4, ST, OUT>(p, ksplit, stream);
    if (p.M <= 48) return launch_variant<3, RF, 2, 1, 4, ST, OUT>(p, ksplit, stream);
    // (four blocks of activation rows for four pairs of wavefronts: no sums to add up at the end, 14.0 against 14.6 us)
    if constexpr (OUT != WideOut::kPartials) return launch_variant<4, RF, 2, 4, 1, ST, OUT>(p, ksplit, stream);
    return launch_variant<4, RF, 2, 1, 4, ST, OUT>(p, ksplit, stream);
}

// y[m][n] = bf16(sum over splits of part[s][m][n]) (+ residual, with the rounding of a separate
// bf16 addition): the split-K linear finished on its own, for callers with no elementwise
// operator to fold the sum into.  Eight outputs per lane.
__global__ void __launch_bounds__(256)
linear_splitk_finish_kernel(const float* __restrict__ part, int ksplit, int64_t split_stride,
                            const uint16_t* __restrict__ res, uint16_t* __restrict__ y, int N, int64_t y_stride) {
    const int vi = int(blockIdx.x) * 256 + threadIdx.x;   // blockIdx.y is the activation row
    if (vi >= N / 8) return;
    const int m = blockIdx.y;
    const int n = vi * 8;
    uint4 o = sum_splits_bf16x8(part + int64_t(m) * N + n, ksplit, split_stride);
    if (res) {
        float a[8], b[8];
        unpack8(o, a);
        unpack8(load16(res + int64_t(m) * y_stride + n), b);
        o.x = pack_bf16x2(a[0] + b[0], a[1] + b[1]);
        o.y = pack_bf16x2(a[2] + b[2], a[3] + b[3]);
        o.z = pack_bf16x2(a[4] + b[4], a[5] + b[5]);
        o.w = pack_bf16x2(a[6] + b[6], a[7] + b[7]);
    }
    store16(y + int64_t(m) * y_stride + n, o);
}

// Partial products of operands whose rows lie too far apart for the 32-bit offsets of the loads above (a column of a
// tensor of tens of gigabytes): a wavefront per output, split after split.
__global__ void __launch_bounds__(kWaveSize)
linear_splitk_far_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, float* __restrict__ part, int K,
                         int64_t x_stride, int64_t w_stride, int ksplit, int chunks_per_split) {
    const int n = int(blockIdx.x), m = int(blockIdx.y), N = int(gridDim.x), M = int(gridDim.y);
    x += m * x_stride;
    w += n * w_stride;
    for (int s = 0; s < ksplit; ++s) {
        const int64_t end = min(int64_t(K), int64_t(s + 1) * chunks_per_split * kWideChunk);
        float sum = 0.f;
        for (int64_t k = int64_t(s) * chunks_per_split * kWideChunk + int(threadIdx.x) * 8; k < end; k += kWaveSize * 8) {
            float a[8], b[8];
            unpack8(load16(x + k), a);
            unpack8(load16(w + k), b);
#pragma unroll
            for (int i = 0; i < 8; ++i) sum = fmaf(a[i], b[i], sum);
        }
        sum = wave_sum(sum);
        if (threadIdx.x == 0) part[(int64_t(s) * M + m) * N + n] = sum;
    }
}

int chunks_of(int K) { return K / kWideChunk; }

// Splits of K of the partial-product form (which imply the weight rows per workgroup, launch_linear_splitk).  One workgroup per compute unit at most:
// with deep rings only one fits a unit, and a second round of a few workgroups costs as much as the first (4096 x
// 14336: 14 splits, 896 workgroups 33 us; 4 splits, 256 workgroups 24 us).  64 rows share an activation tile
// better (2048 x 8192: 9.9 us against 11.3 with 32); with a short K half the splits are worth more, to
// the operator that adds them up as well (2048 x 2048: 32 rows in 4 splits 5.0 us, 64 rows in 8 splits 5.6 us).
int rows_plan(int N, int K, int num_cus) {
    const int rows = chunks_of(K) <= 16 ? 32 : 64;
    const int groups = (N + rows - 1) / rows;
    const int most = std::max(1, std::min(chunks_of(K), num_cus / groups));
    const int per = (chunks_of(K) + most - 1) / most;
    return (chunks_of(K) + per - 1) / per;
}

WideParams wide_params(const uint16_t* x, const uint16_t* w, int M, int N, int K, int64_t x_stride, int64_t w_stride) {
    WideParams p;
    p.x = x;
    p.w0 = p.w1 = w;
    p.res = nullptr;
    p.y = nullptr;
    p.part = nullptr;
    p.M = M; p.N = N; p.K = K;
    p.x_pitch = uint32_t(x_stride * 2);
    p.w_pitch = uint32_t(w_stride * 2);
    p.y_stride = N;
    p.qkv = QkvTarget{};
    return p;
}

}  // namespace

int launch_linear_splitk_finish(const float* part, int ksplit, const uint16_t* res, uint16_t* y, int M, int N,
                                int64_t y_stride, hipStream_t stream) {
    return enqueue(linear_splitk_finish_kernel, dim3(unsigned((N / 8 + 255) / 256), unsigned(M)), dim3(256), 0,
                   stream, part, ksplit, int64_t(M) * N, res, y, N, y_stride);
}

// Splits of K without regard to the activation rows: 128, 256, 512 k per split (1024 for matrices of few rows), the
// largest that still gives about one workgroup of 128 (64) rows per compute unit.
static bool splitk_half_rows(int N, int num_cus) { return (N + 127) / 128 < num_cus / 4; }
int linear_splitk_plan(int N, int K, int num_cus) {
    const int rows_per_wg = splitk_half_rows(N, num_cus) ? 64 : 128;
    const int row_groups = (N + rows_per_wg - 1) / rows_per_wg;
    int per = splitk_half_rows(N, num_cus) ? 8 : 4;
    while (per > 1 && int64_t(row_groups) * ((chunks_of(K) + per - 1) / per) < (3 * int64_t(num_cus)) / 4) per /= 2;
    return (chunks_of(K) + per - 1) / per;
}
// A matrix whose rows alone fill the device has no use for splits (launch_linear_wide): the finer cut, for whoever asks.
int linear_splitk_rows_plan(int N, int K, int num_cus) {
    return (N + 63) / 64 >= num_cus ? linear_splitk_plan(N, K, num_cus) : rows_plan(N, K, num_cus);
}
// Chunks of 128 k a split may cover: what that plan allows, or what the plan above asks for where that is more.
int linear_splitk_max_chunks(int N, int K, int num_cus) {
    const int ks = linear_splitk_rows_plan(N, K, num_cus);
    return std::max(splitk_half_rows(N, num_cus) ? 8 : 4, (chunks_of(K) + ks - 1) / ks);
}

int launch_linear_splitk(const uint16_t* x, const uint16_t* w, float* part, int M, int N, int K, int64_t x_stride,
                         int64_t w_stride, int ksplit, int num_cus, hipStream_t stream) {
    if (M == 1) x_stride = K;   // (a single row has no next one)
    if (x_stride > L3_LINEAR_WIDE_MAX_STRIDE || w_stride > L3_LINEAR_WIDE_MAX_STRIDE) {
        return enqueue(linear_splitk_far_kernel, dim3(unsigned(N), unsigned(M)), dim3(kWaveSize), 0, stream, x, w, part, K, x_stride,
                       w_stride, ksplit, (chunks_of(K) + ksplit - 1) / ksplit);
    }
    WideParams p = wide_params(x, w, M, N, K, x_stride, w_stride);
    p.part = part;
    const int64_t wgs64 = int64_t((N + 63) / 64) * ksplit;
    if (wgs64 * 4 < int64_t(num_cus) * 3) return launch_by_rows<1, 4, WideOut::kPartials>(p, ksplit, stream);
    // more than one workgroup per unit: rings of two stages, so that two fit
    if (wgs64 > num_cus) return launch_by_rows<2, 2, WideOut::kPartials>(p, ksplit, stream);
    return launch_by_rows<2, 4, WideOut::kPartials>(p, ksplit, stream);
}

// The qkv projection of a decode step with rotary embedding and cache append behind it: no splits, so that the sums
// are whole where they are rotated.  32 weight rows per workgroup leave most units idle at one workgroup per row
// group, and the activations, not the weights, are most of what such a workgroup loads: so the activation rows are dealt
// to 16, 32 or 64 per workgroup, as few as the units have room for (the groups of a weight row share an XCD's L2).
// A second round of workgroups costs more than it saves.  Split-K linear and the append that adds it up, one launch with
// 64 / 32 / 16 rows per workgroup, us: 3072 x 2048, 17 rows 7.9, 7.2 / 7.2 / 6.4, 32 rows 8.2, 8.0 / 7.7 / 7.2, 64 rows 9.6,
// 9.9 / 7.8 / 11.0; 6144 x 4096, 32 rows 14.7, - / 13.5 / 21.1, 64 rows 17.9, 17.5 / 22.6 / 30.6.  Up to 16 rows (against the
// skinny kernel's epilogue): 3072 x 2048, 5 rows 6.7, 6.4, 16 rows 7.8, 7.4; 6144 x 4096, 16.4, 10.9 and 20.7, 12.6.
int launch_linear_wide_qkv(const uint16_t* x, const uint16_t* w, const QkvTarget& target, int M, int N, int K, int64_t x_stride,
                           int64_t w_stride, int num_cus, hipStream_t stream) {
    WideParams p = wide_params(x, w, M, N, K, x_stride, w_stride);
    p.qkv = target;
    const int row_groups = (N + 31) / 32;
    auto room = [&](int rows) { return M <= rows || row_groups * ((M + rows - 1) / rows) <= num_cus; };
    if (room(16)) return launch_variant<1, 1, 2, 1, 4, 6, WideOut::kQkv>(p, (M + 15) / 16, stream);
    if (room(32)) return launch_variant<2, 1, 2, 1, 4, 4, WideOut::kQkv>(p, (M + 31) / 32, stream);
    if (M <= 48) return launch_variant<3, 1, 2, 1, 4, 6, WideOut::kQkv>(p, 1, stream);
    return launch_variant<4, 1, 2, 1, 4, 6, WideOut::kQkv>(p, 1, stream);
}

// The whole sums in one launch: y, or with w_up the SwiGLU product, plus the residual if there is one.
int launch_linear_wide(const uint16_t* x, const uint16_t* w, const uint16_t* w_up, const uint16_t* res, uint16_t* y, int M,
                       int N, int K, int64_t x_stride, int64_t w_stride, int64_t y_stride, int num_cus, hipStream_t stream) {
    WideParams p = wide_params(x, w, M, N, K, x_stride, w_stride);
    p.res = res;
    p.y = y;
    p.y_stride = y_stride;
    if (w_up) {
        p.w1 = w_up;
        // one workgroup per unit with a deep ring, or two with a shallow one (14336 x 4096, 448 workgroups: 48.2 -> 44.4 us)
        if ((N + 31) / 32 > num_cus) return launch_by_rows<2, 2, WideOut::kSwiglu>(p, 1, stream);
        return launch_by_rows<2, 4, WideOut::kSwiglu>(p, 1, stream);
    }
    if (N < 128 * num_cus) {   // fewer than 128 rows per unit: workgroups of 64
        return (N + 63) / 64 > num_cus ? launch_by_rows<2, 2, WideOut::kRows>(p, 1, stream)
                                       : launch_by_rows<2, 4, WideOut::kRows>(p, 1, stream);
    }
    if (M <= 16) return launch_variant<1, 1, 8, 1, 1, 2, WideOut::kRows>(p, 1, stream);
    if (M <= 32) return launch_variant<2, 2, 4, 2, 1, 2, WideOut::kRows>(p, 1, stream);
    return launch_variant<4, 2, 2, 4, 1, 2, WideOut::kRows>(p, 1, stream);
}

}  // namespace l3
