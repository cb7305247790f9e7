// All transformer layers of one decode step for up to four sequences in ONE launch (model.py:143-150, :92-122, :134
// for T = 1): what at batch 1 is otherwise five launches per layer, each with a ramp, a tail and a dependent
// launch's 1.7 us between them.
//
// What bounds it is the stream over the weights (1.95 GB at the 1B shape), so the kernel is built around not letting that
// stream stop.  One workgroup per compute unit stays for the whole step.  Two of its ten wavefronts only load:
// they keep a ring of seven 16 KiB weight stages in LDS full, in the order the stages will be needed, across
// every synchronisation -- while the other eight wait for activations, the next 28 MB of weights arrive.
//
// Sixteen layers at 256 cached tokens and 1 / 2 / 3 / 4 rows: 386 / 428 / 463 / 492 us (5.0 TB/s at one row), recorded
// launches per operator 559 / 589 / 637 / 679 us.  A layer's 24 us are 18 us of stream and 6 us in which it waits for the
// chain of hand-overs.  Fetching further ahead into the L2 made everything slower (431 -> 484 us, the
// polls and the ring's loads queue behind the fetches), a ring of six stages costs 0.4 %.
//
// The work is laid over the eight XCDs the way tensor parallelism lays it over GPUs.  XCD g owns kv head g: its rows
// of c_attn, the attention of its query heads, the k columns of c_proj those feed, an eighth of the hidden
// units of the MLP, and the k columns of the down projection those feed.  So only the two places where a layer
// sums over everything (behind c_proj and behind the down projection) cross XCDs, as float32 partial rows that every
// XCD adds up in the same order; all other hand-overs stay behind one L2.
// What one workgroup hands to others carries its own tag, so that nobody waits for an acknowledgement, a counter and a
// flag one after the other: inside an XCD 32-bit words of a bf16 value, the launch's number and the writer's XCD, plain stores,
// polled past the L1 (0.6 us for a row of 2048 to all 32 workgroups; a counter in the L2 and then the data 1.5 us); across XCDs 64-bit words
// of a float32 value and the launch's and the layer's number, device-scope stores and polls (1.3 us; a flag per XCD behind
// an L2 counter and then the data 2.3 us, one counter 3.5 us).  Every place is written once per launch, or per layer and
// again only after all its readers have handed in something later.
//
// Every wait is bounded.  A wavefront whose wait runs out (the launch shares the device with something that keeps
// part of it from becoming resident, or workgroups are not placed on XCDs in turn) raises the error word of the
// control block and goes on without waiting, so that the launch always ends; the caller looks at the word when it
// reads results, discards them and does the work again with the launches per operator.
//
// Rounding points are those of the separate operators.
#include "attn_merge.hpp"
#include "lds_loads.hpp"

namespace l3 {

namespace {

// The 1B architecture: hidden 2048, 32 / 8 heads of 64, 8192 hidden units.
constexpr int kC = 2048, kH = 8192, kHD = 64, kR = 4, kKVH = 8;
constexpr int kXcds = 8, kSlots = 32;                      // workgroups: XCD g = id % 8, slot s = id / 8
constexpr int kComputeWaves = 8, kRingWaves = 2;
constexpr int kLayersThreads = (kComputeWaves + kRingWaves) * kWaveSize;
constexpr int kStageBytes = 16 << 10, kStages = 7;         // 64 pieces of four rows x 128 k
constexpr int kQkvRows = (kR + 2) * kHD / kSlots;          // 12 rows of c_attn per workgroup (of its XCD's 384) ...
constexpr int kQkvStages = 3;                              // ... with all of k: 48 pieces
constexpr int kProjStages = kR * kHD / 128;                // 64 rows x the 256 k of the XCD's heads
constexpr int kMlpStages = kC / 128;                       // 32 gate and 32 up rows x all of k
constexpr int kDownStages = kH / kXcds / 128;              // 64 rows x the 1024 k of the XCD's hidden units
constexpr int kLayerStages = kQkvStages + kProjStages + kMlpStages + kDownStages;
constexpr int kWaitPolls = 1 << 15;                        // about 15 ms
static_assert(kQkvRows % 4 == 0 && kHD % 4 == 0 && kC / kSlots == 64 && kH / kXcds / kSlots == 32, "pieces of four rows");

struct LayersParams {
    const DecodeLayerPointers* layers;
    const uint16_t* x;          // (M, C), or with tokens the embedding (vocab, C) they pick the rows from
    const int64_t* tokens;
    int64_t token_stride, vocab;
    uint16_t* out;              // (M, C)
    const float* rope_table;
    const int* pos;
    unsigned char* ws;          // control block, then exchange buffers
    int64_t c_sb, c_st;
    int n_layer, cache_len, table_rows;
    float eps, scale_log2e;
};

// Control block: all words zero before the first launch.
struct Control {
    unsigned error[64];      // [0] != 0: a wait ran out
    unsigned launches[64];   // [0] so far; the number of a launch is its tag
};
static_assert(sizeof(Control) <= kDecodeLayersControlBytes, "control block");

__device__ __forceinline__ void store_device(unsigned* p, unsigned v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned load_device(const unsigned* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_device(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t load_device(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Row m of the input.
__device__ __forceinline__ const uint16_t* input_row(const LayersParams& p, int m) {
    int64_t row = m;
    if (p.tokens) row = max(int64_t(0), min(p.tokens[m * p.token_stride], p.vocab - 1));
    return p.x + row * kC;
}
__device__ __forceinline__ void wait_own_accesses() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// two tagged bf16 values
__device__ __forceinline__ bool tags_are(uint64_t v, uint32_t tag) {
    return ((uint32_t(v) ^ tag) & 0xffffu) == 0 && ((uint32_t(v >> 32) ^ tag) & 0xffffu) == 0;
}
__device__ __forceinline__ float tagged_lo(uint64_t v) { return __uint_as_float(uint32_t(v) & 0xffff0000u); }
__device__ __forceinline__ float tagged_hi(uint64_t v) { return __uint_as_float(uint32_t(v >> 32) & 0xffff0000u); }
__device__ __forceinline__ uint32_t tagged_pair(uint64_t v) { return (uint32_t(v) >> 16) | (uint32_t(v >> 32) & 0xffff0000u); }
__device__ __forceinline__ float round_bf16(float v) { return __uint_as_float(f32_to_bf16_bits(v) << 16); }

// A layer's pointers, read through the scalar cache (the table does not change while a launch runs).
__device__ __forceinline__ const __attribute__((address_space(4))) DecodeLayerPointers& scalar_layer(const DecodeLayerPointers* layers, int i) {
    return ((const __attribute__((address_space(4))) DecodeLayerPointers*)(layers))[i];
}

// The loading wavefronts.  A stage is 16 pieces of four rows x 256 bytes: for the qkv rows four rows with all of k (a
// piece per 128 k), otherwise 64 rows x 128 k; every loading wavefront has its share of them.  In the ring the
// 16-byte chunk c of row r of a 16-row block sits at position c ^ (r & 15).
//
// They go through the same barriers as the compute wavefronts.  Before a barrier that makes a stage ready they
// wait for their part of it; behind each barrier they refill the places of the stages that everybody has multiplied.
// What happens at which barrier of a layer is known at compile time, and so is unrolled: with the stage as a run-time
// state its hundred or two scalar instructions took longer (0.6 to 1 us) than its bytes do.
struct LayerSchedule {
    // barriers of a layer: sums of squares, qkv ready, its sums, its results; attention's parts
    static constexpr int kBeforeProj = 5;
    static constexpr int kBeforeMlp = kBeforeProj + kProjStages + 3;   // then one per stage, behind the products, behind the
    static constexpr int kBeforeDown = kBeforeMlp + kMlpStages + 2;    // hand-over, and before the gate and up stages one more
    static constexpr int kBarriers = kBeforeDown + kDownStages + 2;
    static constexpr int in_phase(int e) { return e - (e < kBeforeMlp ? kBeforeProj : e < kBeforeDown ? kBeforeMlp : kBeforeDown); }
    static constexpr int stages(int e) { return e < kBeforeMlp ? kProjStages : e < kBeforeDown ? kMlpStages : kDownStages; }
    static constexpr int first(int e) {
        return e < kBeforeMlp ? kQkvStages : e < kBeforeDown ? kQkvStages + kProjStages : kQkvStages + kProjStages + kMlpStages;
    }
    // the stages below are behind everybody at barrier e
    static constexpr int freed(int e) {
        if (e < kBeforeProj) return e <= 2 ? 0 : kQkvStages;   // (not before the hand-over of q, k and v, which would queue behind the loads)
        return first(e) + (in_phase(e) < stages(e) ? in_phase(e) : stages(e));
    }
    // the stage (with those before it) that must have landed at barrier e, or -1
    static constexpr int ready(int e) {
        if (e < kBeforeProj) return e == 1 ? kQkvStages - 1 : -1;
        return in_phase(e) < stages(e) ? freed(e) : -1;
    }
    static constexpr int requested(int e) { return (e < 0 ? 0 : freed(e)) + kStages; }   // stages, behind barrier e
};

// One loading wavefront: its pieces of each stage, into the ring.
struct RingLoader {
    static constexpr int kPieces = 16 / kRingWaves;
    const char *qkv, *proj, *mlp, *down, *qkv_n, *proj_n, *mlp_n, *down_n;   // its rows in this layer's weights and the next's
    int64_t proj_at, mlp_at, down_at;
    int qkv_row[kQkvStages];
    int s, place = 0;
    bool up;   // its rows of the gate and up stages are w_up's
    uint32_t ring, half, lane16, row;

    __device__ __forceinline__ RingLoader(uint32_t s_ring, int g, int slot, int lw) {
        const int lane = threadIdx.x & (kWaveSize - 1);
        const int first_row = lw * kPieces * 4;
        s = slot;
        ring = s_ring + uint32_t(lw * kPieces * 1024);
        half = uint32_t(lw * kPieces * 256);
        lane16 = uint32_t(((lane & 15) ^ (lane >> 4)) * 16);
        row = uint32_t(lane >> 4);
#pragma unroll
        for (int i = 0; i < kQkvStages; ++i) {
            const int r = s * kQkvRows + i * 4;   // of the XCD's q | k | v rows
            qkv_row[i] = r < kR * kHD ? g * (kR * kHD) + r
                : r < (kR + 1) * kHD ? kKVH * kR * kHD + g * kHD + r - kR * kHD
                                     : kKVH * (kR + 1) * kHD + g * kHD + r - (kR + 1) * kHD;
        }
        up = first_row >= 32;   // gate rows in the first half of a stage, up rows behind
        proj_at = int64_t(s * 64 + first_row) * (kC * 2) + g * (kR * kHD * 2);
        mlp_at = int64_t(g * (kH / kXcds) + s * 32 + first_row % 32) * (kC * 2);
        down_at = int64_t(s * 64 + first_row) * (kH * 2) + g * (kH / kXcds * 2);
    }
    __device__ __forceinline__ void read_next(const DecodeLayerPointers* layers, int l) {
        const auto& L = scalar_layer(layers, l);
        qkv_n = reinterpret_cast<const char*>(L.c_attn);
        proj_n = reinterpret_cast<const char*>(L.c_proj) + proj_at;
        mlp_n = reinterpret_cast<const char*>(up ? L.w_up : L.w_gate) + mlp_at;
        down_n = reinterpret_cast<const char*>(L.w_down) + down_at;
    }
    __device__ __forceinline__ void next_layer() {
        qkv = qkv_n;
        proj = proj_n;
        mlp = mlp_n;
        down = down_n;
    }
    // Stage I of this layer (from kLayerStages on: of the next).  Workgroups start the long phases at different k.
    template <int I>
    __device__ __forceinline__ void request() {
        constexpr bool NEXT = I >= kLayerStages;
        constexpr int J = NEXT ? I - kLayerStages : I;
        constexpr bool QKV = J < kQkvStages, DOWN = J >= kLayerStages - kDownStages;
        constexpr int PITCH = DOWN ? kH * 2 : kC * 2;
        const char* base;
        int koff = 0;
        if constexpr (QKV) {
            base = (NEXT ? qkv_n : qkv) + int64_t(qkv_row[J]) * PITCH;
        } else if constexpr (J < kQkvStages + kProjStages) {
            base = NEXT ? proj_n : proj;
            koff = (J - kQkvStages) * 256;
        } else if constexpr (!DOWN) {
            base = NEXT ? mlp_n : mlp;
            koff = (J - kQkvStages - kProjStages + s) % kMlpStages * 256;
        } else {
            base = NEXT ? down_n : down;
            koff = (J - kQkvStages - kProjStages - kMlpStages + s) % kDownStages * 256;
        }
        const srd_t srd = make_srd(base);
        const uint32_t lds = ring + uint32_t(place) * kStageBytes;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const uint32_t piece = QKV ? (lane16 ^ uint32_t(J << 6)) + half + uint32_t(i * 256)
                                       : (lane16 ^ uint32_t((i & 3) << 6)) + uint32_t(i * 4 * PITCH);
            load_to_lds<true>(srd, lds + uint32_t(i * 1024), piece + row * uint32_t(PITCH), koff);
        }
        place = place == kStages - 1 ? 0 : place + 1;
    }
    template <int E>
    __device__ __forceinline__ void before_barrier(bool more) {
        constexpr int issued = LayerSchedule::requested(E - 1), ready = LayerSchedule::ready(E);
        if constexpr (ready >= 0) {
            constexpr int last = issued < kLayerStages ? issued : kLayerStages;
            if (issued <= kLayerStages || more) wait_loads<kPieces * (issued - ready - 1)>();
            else wait_loads<kPieces * (last - ready - 1)>();
        }
    }
};

// stages LO .. HI - 1; `more`: there is a next layer
template <int LO, int HI>
__device__ __forceinline__ void request_all(RingLoader& l, bool more) {
    if constexpr (LO < HI) {
        if (LO < kLayerStages || more) l.request<LO>();
        request_all<LO + 1, HI>(l, more);
    }
}
template <int E>
__device__ __forceinline__ void barriers_from(RingLoader& l, bool more) {
    if constexpr (E < LayerSchedule::kBarriers) {
        l.before_barrier<E>(more);
        barrier();
        request_all<LayerSchedule::requested(E - 1), LayerSchedule::requested(E)>(l, more);
        barriers_from<E + 1>(l, more);
    }
}
__device__ __forceinline__ void load_into_ring(const LayersParams& p, RingLoader l) {
    l.read_next(p.layers, 0);
    l.next_layer();
    request_all<0, kStages>(l, true);
#pragma unroll 1
    for (int layer = 0; layer < p.n_layer; ++layer) {
        l.read_next(p.layers, min(layer + 1, p.n_layer - 1));
        barriers_from<0>(l, layer + 1 < p.n_layer);
        l.next_layer();
    }
}

template <int M>
__global__ void __launch_bounds__(kLayersThreads)
decode_layers_kernel(const LayersParams p) {
    constexpr int HP = kC * 2 + 16, TP = kH / kXcds * 2 + 16, YP = kR * kHD * 2 + 16;   // LDS row pitches in bytes
    using Tile = MfmaTile<kHD, 4>;
    __shared__ __align__(1024) unsigned char s_ring[kStages * kStageBytes];
    // the attention slabs (behind the last tile a wavefront's output rows lie in its own), and at other times the layer's input rows and hidden units
    __shared__ __align__(16) unsigned char s_act[kComputeWaves * Tile::SLAB];
    static_assert(M * (HP + TP) <= kComputeWaves * Tile::SLAB, "activations in the slabs");
    __shared__ __align__(16) unsigned char s_y[M * YP];
    __shared__ float s_m[kComputeWaves][kR], s_l[kComputeWaves][kR];
    __shared__ float s_red[kComputeWaves * 16 * 4], s_squares[kComputeWaves][M];
    __shared__ __align__(16) uint32_t s_q[M * kR * kHD / 2];
    auto s_o = [&](int w, int h) { return reinterpret_cast<float*>(s_act + w * Tile::SLAB) + h * kHD; };
    static_assert(kR * kHD * 4 <= Tile::SLAB, "output rows in the slab");
    unsigned char* const s_h = s_act;
    unsigned char* const s_t = s_act + M * HP;

    int lane = threadIdx.x & (kWaveSize - 1);
    const int wave = wave_uniform(int(threadIdx.x) / kWaveSize);
    int fn = lane & 15, fg = lane >> 4;
    const int g = wave_uniform(int(blockIdx.x) % kXcds), s = wave_uniform(int(blockIdx.x) / kXcds);
    const bool loads = wave >= kComputeWaves;
    Control* const ctl = reinterpret_cast<Control*>(p.ws);
    // exchange buffers: two float32 partial rows per XCD; per layer and XCD the rows its workgroups hand each other
    uint64_t* const part = reinterpret_cast<uint64_t*>(p.ws + kDecodeLayersControlBytes);   // [2][XCD][M][C]
    uint32_t* const local = reinterpret_cast<uint32_t*>(part + 2 * kXcds * M * kC);
    constexpr int kQkv = (kR + 2) * kHD;
    constexpr int kLocal = M * (2 * kC + kQkv + kH / kXcds);   // x, x behind c_proj, q | k | v, hidden units

    if (loads) {
        load_into_ring(p, RingLoader(lds_address(s_ring), g, s, wave - kComputeWaves));
        return;
    }
    auto sync = []() __attribute__((always_inline)) { barrier_after_lds(); };

    // ---- waiting for other workgroups: poll() until it says that everything it reads is there
    const uint32_t launch = uint32_t(wave_uniform(int(ctl->launches[0]))) + 1;
    // A word handed over inside the XCD names its launch and the XCD that wrote it, and is awaited with the reader's own: from
    // a workgroup that runs elsewhere than its number says nothing is taken, its K/V row (no tag of its own) included.
    const uint32_t tag = (launch & 0xfffu) << 4 | xcc_id();
    bool alone = wave_uniform(int(load_device(&ctl->error[0]))) != 0;   // a wait has run out: go on without waiting
    auto wait_for = [&](auto poll) __attribute__((always_inline)) {
        for (int polls = 1; __builtin_amdgcn_ballot_w64(!poll()) != 0 && !alone; ++polls) {
            if (polls % 1024 == 0 && (polls >= kWaitPolls || wave_uniform(int(load_device(&ctl->error[0]))) != 0)) {
                alone = true;
                if (lane == 0) store_device(&ctl->error[0], 1u);
            }
        }
    };
    auto tagged = [&](float v) __attribute__((always_inline)) { return (f32_to_bf16_bits(v) << 16) | tag; };

    // ---- arithmetic of the compute wavefronts
    // 32 k of a stage that holds 64 rows x 128 k: rows 16 (wave % 4) .., k steps 2 (wave / 4) and + 1 of the stage
    auto multiply = [&](int slot, const unsigned char* act, int pitch, int chunk, f32x4_t& acc) __attribute__((always_inline)) {
        const int row = (wave & 3) * 16 + fn;
        const unsigned char* a_row = s_ring + slot * kStageBytes + row * 256;
        const unsigned char* b_row = act + min(fn, M - 1) * pitch + chunk * 256 + fg * 16;   // columns past M are not used
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int ks = (wave >> 2) * 2 + i;
            const uint4 a = *reinterpret_cast<const uint4*>(a_row + (((ks * 4 + fg) ^ fn) * 16));
            const uint4 b = *reinterpret_cast<const uint4*>(b_row + ks * 64);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), acc,
                                                          0, 0, 0);
        }
    };
    // the two k halves of 64 rows meet in s_red[half][row][m]
    auto hand_in = [&](const f32x4_t& acc) __attribute__((always_inline)) {
        if (fn < M) {
#pragma unroll
            for (int r = 0; r < 4; ++r) s_red[((wave >> 2) * 64 + (wave & 3) * 16 + 4 * fg + r) * 4 + fn] = acc[r];
        }
    };
    auto row_sum = [&](int row, int m) { return s_red[row * 4 + m] + s_red[(64 + row) * 4 + m]; };
    // RMSNorm of M rows into s_h, an eighth per wavefront: rows that the XCD's workgroups hand over, or (first) the input
    auto normalise = [&](const uint32_t* rows, bool first, const uint16_t* weight) __attribute__((always_inline)) {
        const int col = (wave * kWaveSize + lane) * 4;
        const uint2 gw = *reinterpret_cast<const uint2*>(weight + col);
        float f[M][4];
        if (first) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const uint2 v = *reinterpret_cast<const uint2*>(input_row(p, m) + col);
                f[m][0] = __uint_as_float(v.x << 16);
                f[m][1] = __uint_as_float(v.x & 0xffff0000u);
                f[m][2] = __uint_as_float(v.y << 16);
                f[m][3] = __uint_as_float(v.y & 0xffff0000u);
            }
        } else {
            uint64_t v[M][2];
            wait_for([&]() {
                bool there = true;
#pragma unroll
                for (int m = 0; m < M; ++m) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) v[m][i] = load_device(reinterpret_cast<const uint64_t*>(rows + m * kC + col) + i);
                }
#pragma unroll
                for (int m = 0; m < M; ++m) there = there && tags_are(v[m][0], tag) && tags_are(v[m][1], tag);
                return there;
            });
#pragma unroll
            for (int m = 0; m < M; ++m) {
                f[m][0] = tagged_lo(v[m][0]);
                f[m][1] = tagged_hi(v[m][0]);
                f[m][2] = tagged_lo(v[m][1]);
                f[m][3] = tagged_hi(v[m][1]);
            }
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            float ss = f[m][0] * f[m][0];
#pragma unroll
            for (int i = 1; i < 4; ++i) ss = fmaf(f[m][i], f[m][i], ss);
            ss = wave_sum(ss);
            if (lane == 0) s_squares[wave][m] = ss;
        }
        sync();
        const float w0 = __uint_as_float(gw.x << 16), w1 = __uint_as_float(gw.x & 0xffff0000u);
        const float w2 = __uint_as_float(gw.y << 16), w3 = __uint_as_float(gw.y & 0xffff0000u);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            float ss = s_squares[0][m];
#pragma unroll
            for (int w = 1; w < kComputeWaves; ++w) ss += s_squares[w][m];
            const float inv = rsqrtf(ss / float(kC) + p.eps);
            uint2 o;
            o.x = pack_bf16x2(f[m][0] * inv * w0, f[m][1] * inv * w1);
            o.y = pack_bf16x2(f[m][2] * inv * w2, f[m][3] * inv * w3);
            *reinterpret_cast<uint2*>(s_h + m * HP + col * 2) = o;
        }
    };

    const int pos = wave_uniform(*p.pos);
    const int kv_len = max(1, min(pos + 1, p.cache_len));
    const bool pos_ok = pos >= 0 && pos < p.cache_len && pos < p.table_rows;
    // wavefront m < M: column 64 s + lane of row m of the residual stream (a bf16 value)
    float xcol = wave < M ? bf16_to_f32(input_row(p, wave)[s * 64 + lane]) : 0.f;
    // The XCDs' partial sums of row m = wave join it; every XCD gets the new row (dst, its own copy).
    auto join = [&](uint64_t* rows, uint32_t layer_tag, uint32_t* dst) __attribute__((always_inline)) {
        uint64_t* const at = rows + wave * kC + s * 64 + lane;
        store_device(at + g * (M * kC), uint64_t(layer_tag) << 32 | __float_as_uint(row_sum(lane, wave)));
        uint64_t v[kXcds];
        wait_for([&]() {
            bool there = true;
#pragma unroll
            for (int j = 0; j < kXcds; ++j) v[j] = load_device(at + j * (M * kC));
#pragma unroll
            for (int j = 0; j < kXcds; ++j) there = there && uint32_t(v[j] >> 32) == layer_tag;
            return there;
        });
        float r = __uint_as_float(uint32_t(v[0]));
#pragma unroll
        for (int j = 1; j < kXcds; ++j) r += __uint_as_float(uint32_t(v[j]));
        xcol = round_bf16(xcol + round_bf16(r));
        if (dst) dst[wave * kC + s * 64 + lane] = tagged(xcol);
    };
    // What the layer reads besides its weights comes into the L2 while somebody else is waited for: a workgroup fetches
    // its part of the lines (past the L1, which must not hold them).
    auto fetch = [&](int layer, int first_wave) __attribute__((always_inline)) {
        const auto& L = scalar_layer(p.layers, layer);
        const int id = int(threadIdx.x) - first_wave * kWaveSize, ids = (kComputeWaves - first_wave) * kWaveSize;
        unsigned got = 0;
        if (id < 4) {
            const uint16_t* w = (id & 1) ? L.ln_2 : L.ln_1;
            got = load_device(reinterpret_cast<const unsigned*>(w + s * 64 + (id >> 1) * 32));
        }
        const int rows = min(pos, p.cache_len);
        for (int i = id * kSlots + s; i < M * rows; i += ids * kSlots) {
            const int64_t cell = int64_t(i / rows) * p.c_sb + int64_t(i % rows) * p.c_st + g * kHD;
            got ^= load_device(reinterpret_cast<const unsigned*>(L.cache_k + cell)) ^ load_device(reinterpret_cast<const unsigned*>(L.cache_v + cell)) ^
                   load_device(reinterpret_cast<const unsigned*>(L.cache_k + cell + 32)) ^ load_device(reinterpret_cast<const unsigned*>(L.cache_v + cell + 32));
        }
        asm volatile("" ::"v"(got));
    };
    // this lane's pair of a q or k row (wavefront 0, below)
    float2 cs = make_float2(1.f, 0.f);
    constexpr int PAIRS = kQkvRows / 2;
    if (pos_ok) cs = *reinterpret_cast<const float2*>(p.rope_table + int64_t(pos) * kHD + (s * kQkvRows + 2 * (lane % PAIRS)) % kHD);
    fetch(0, 0);

    int slot = 0;   // ring place of the stage multiplied next
    auto next_slot = [&]() {
        const int now = slot;
        if (++slot == kStages) slot = 0;
        return now;
    };
#pragma unroll 1
    for (int layer = 0; layer < p.n_layer; ++layer) {
        // (addresses worked out where they are used: kept over the layers they would not fit into the registers)
        asm volatile("" : "+v"(lane), "+v"(fn), "+v"(fg));
        const auto& L = scalar_layer(p.layers, layer);
        uint32_t* const lx = local + (int64_t(layer) * kXcds + g) * kLocal;     // written by the layer before
        uint32_t* const lmid = lx + M * kC;
        uint32_t* const lqkv = lmid + M * kC;
        uint32_t* const lt = lqkv + M * kQkv;
        const uint32_t layer_tag = (launch << 16) + uint32_t(layer) + 1;

        // ---- q, k and v of the XCD's head: 12 rows per workgroup, k dealt to the wavefronts
        normalise(lx, layer == 0, L.ln_1);
        sync();
        {
            f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
            const int row = min(fn, kQkvRows - 1);   // (rows past the twelfth are not used)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int chunk = 2 * wave + (i >> 2), ks = i & 3;
                int place = slot + (row >> 2);
                if (place >= kStages) place -= kStages;
                const uint4 a = *reinterpret_cast<const uint4*>(s_ring + place * kStageBytes + chunk * 1024 + (row & 3) * 256 +
                                                                (((ks * 4 + fg) ^ row) * 16));
                const uint4 b = *reinterpret_cast<const uint4*>(s_h + min(fn, M - 1) * HP + chunk * 256 + ks * 64 + fg * 16);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                              acc, 0, 0, 0);
            }
            if (fn < M && fg < kQkvRows / 4) {
#pragma unroll
                for (int r = 0; r < 4; ++r) s_red[(wave * 16 + 4 * fg + r) * 4 + fn] = acc[r];
            }
        }
        slot += kQkvStages;
        if (slot >= kStages) slot -= kStages;
        sync();
        if (wave == 0) {
            const int m = lane / PAIRS, pr = lane % PAIRS;
            if (m < M) {
                float v0 = 0.f, v1 = 0.f;
#pragma unroll
                for (int w = 0; w < kComputeWaves; ++w) {
                    v0 += s_red[(w * 16 + 2 * pr) * 4 + m];
                    v1 += s_red[(w * 16 + 2 * pr + 1) * 4 + m];
                }
                const int r = s * kQkvRows + 2 * pr;                 // of the XCD's q | k | v rows
                uint32_t yw = pack_bf16x2(v0, v1);
                if (r < (kR + 1) * kHD) yw = rotate_pair(yw, cs.x, cs.y);
                if (r >= kR * kHD && pos_ok) {
                    const int64_t cell = m * p.c_sb + int64_t(pos) * p.c_st + g * kHD;
                    uint16_t* const to = r < (kR + 1) * kHD ? L.cache_k + cell + r - kR * kHD : L.cache_v + cell + r - (kR + 1) * kHD;
                    *reinterpret_cast<uint32_t*>(to) = yw;
                    wait_own_accesses();   // it is in the L2 before the word below says so
                }
                *reinterpret_cast<uint64_t*>(lqkv + m * kQkv + r) = uint64_t(yw & 0xffff0000u | tag) << 32 | (yw << 16 | tag);
            }
        }
        if (wave < kQkv / 2 / kWaveSize) {
            uint64_t v[M];
            wait_for([&]() {
                bool there = true;
#pragma unroll
                for (int m = 0; m < M; ++m) v[m] = load_device(reinterpret_cast<const uint64_t*>(lqkv + m * kQkv) + threadIdx.x);
#pragma unroll
                for (int m = 0; m < M; ++m) there = there && tags_are(v[m], tag);
                return there;
            });
            if (threadIdx.x < kR * kHD / 2) {
#pragma unroll
                for (int m = 0; m < M; ++m) s_q[m * (kR * kHD / 2) + threadIdx.x] = tagged_pair(v[m]);
            }
        }
        sync();

        // ---- attention of the XCD's query heads, by every workgroup for itself (at the lengths this kernel is used
        // for the K/V of a head come out of the L2 faster than another hand-over would take); the wavefronts
        // share the rows, and what one has is merged
        {
            const int m = wave % M, part_of_m = wave / M, parts_of_m = (kComputeWaves - m + M - 1) / M;
            bf16x8_t qfrag[Tile::KC];
#pragma unroll
            for (int i = 0; i < Tile::KC; ++i) {
                uint4 qv = make_uint4(0u, 0u, 0u, 0u);
                if (fn < kR) qv = *reinterpret_cast<const uint4*>(&s_q[(m * (kR * kHD) + fn * kHD + (i * 4 + fg) * 8) / 2]);
                qfrag[i] = __builtin_bit_cast(bf16x8_t, qv);
            }
            f32x4_t O[Tile::NB];
#pragma unroll
            for (int nb = 0; nb < Tile::NB; ++nb) O[nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            float m_run = kMaskedScore, l_part = 0.f;
            const int64_t head = m * p.c_sb + g * kHD;
            mfma_tile_loop<kHD, 4>(L.cache_k, L.cache_v, head, head, p.c_st, p.c_st, s_act + wave * Tile::SLAB, qfrag,
                                   part_of_m * Tile::WT, kv_len, parts_of_m * Tile::WT, kv_len, kv_len, p.scale_log2e, O, m_run,
                                   l_part);
            l_part += __shfl_xor(l_part, 16, kWaveSize);
            l_part += __shfl_xor(l_part, 32, kWaveSize);
            if (fn < kR) {
#pragma unroll
                for (int nb = 0; nb < Tile::NB; ++nb) {
                    *reinterpret_cast<float4*>(s_o(wave, fn) + nb * 16 + fg * 4) = make_float4(O[nb][0], O[nb][1], O[nb][2], O[nb][3]);
                }
                if (fg == 0) {
                    s_m[wave][fn] = (m_run == kMaskedScore) ? kMaskedScore : m_run * p.scale_log2e;
                    s_l[wave][fn] = l_part;
                }
            }
        }
        sync();
        if (wave < M * (kR * kHD / 2 / kWaveSize)) {
            const int m = wave / (kR * kHD / 2 / kWaveSize), t = int(threadIdx.x) % (kR * kHD / 2);
            const int h = t / (kHD / 2), d = (t % (kHD / 2)) * 2;
            float top = s_m[m][h];
#pragma unroll
            for (int w = m + M; w < kComputeWaves; w += M) top = fmaxf(top, s_m[w][h]);
            float l = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
            for (int w = m; w < kComputeWaves; w += M) {
                const float e = fast_exp2(s_m[w][h] - top);   // wavefronts without a tile: 0
                l = fmaf(s_l[w][h], e, l);
                o0 = fmaf(s_o(w, h)[d], e, o0);
                o1 = fmaf(s_o(w, h)[d + 1], e, o1);
            }
            const float inv = 1.0f / l;
            *reinterpret_cast<uint32_t*>(s_y + m * YP + (h * kHD + d) * 2) = pack_bf16x2(o0 * inv, o1 * inv);
        }

        // ---- c_proj over the XCD's 256 k: partial sums of 64 rows per workgroup
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int j = 0; j < kProjStages; ++j) {
            sync();
            const int place = next_slot();
            multiply(place, s_y, YP, j, acc);
        }
        hand_in(acc);
        sync();
        if (wave < M) join(part, layer_tag, lmid);
        sync();

        // ---- gate and up: 32 hidden units per workgroup
        normalise(lmid, false, L.ln_2);
        acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int j = 0; j < kMlpStages; ++j) {
            sync();
            const int place = next_slot();
            multiply(place, s_h, HP, (j + s) % kMlpStages, acc);
        }
        hand_in(acc);
        sync();
        if (wave == 0) {
            constexpr int UNITS = kH / kXcds / kSlots;
#pragma unroll
            for (int i = 0; i < (UNITS * M + kWaveSize - 1) / kWaveSize; ++i) {
                const int u = lane % UNITS, m = lane / UNITS + 2 * i;
                if (m < M) {
                    const float gate = round_bf16(row_sum(u, m)), up = round_bf16(row_sum(UNITS + u, m));
                    lt[m * (kH / kXcds) + s * UNITS + u] = tagged(silu_rounded(gate) * up);
                }
            }
        }
        sync();

        // ---- down projection over the XCD's 1024 hidden units
        {
            static_assert(kH / kXcds == 2 * kComputeWaves * kWaveSize, "two hidden units per thread");
            uint64_t v[M];
            wait_for([&]() {
                bool there = true;
#pragma unroll
                for (int m = 0; m < M; ++m) v[m] = load_device(reinterpret_cast<const uint64_t*>(lt + m * (kH / kXcds)) + threadIdx.x);
#pragma unroll
                for (int m = 0; m < M; ++m) there = there && tags_are(v[m], tag);
                return there;
            });
#pragma unroll
            for (int m = 0; m < M; ++m) *reinterpret_cast<uint32_t*>(s_t + m * TP + threadIdx.x * 4) = tagged_pair(v[m]);
        }
        acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int j = 0; j < kDownStages; ++j) {
            sync();
            const int place = next_slot();
            multiply(place, s_t, TP, (j + s) % kDownStages, acc);
        }
        hand_in(acc);
        sync();
        const bool last = layer + 1 == p.n_layer;
        if (wave < M) {
            join(part + kXcds * M * kC, layer_tag, last ? nullptr : lx + kXcds * kLocal);
            if (last && g == 0) p.out[wave * kC + s * 64 + lane] = uint16_t(f32_to_bf16_bits(xcol));
        } else if (!last) {
            fetch(layer + 1, M);
        }
        sync();
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl->launches[0] = launch;   // everybody read it before handing anything in
}

}  // namespace

bool decode_layers_supported(int M, int C, int H, int QH, int KVH, int HD, int num_cus) {
    return M >= 1 && M <= 4 && C == kC && H == kH && QH == kKVH * kR && KVH == kKVH && HD == kHD && num_cus == kXcds * kSlots;
}

size_t decode_layers_workspace_bytes(int M, int n_layer) {
    const size_t part = size_t(2) * kXcds * M * kC * sizeof(uint64_t);
    const size_t local = size_t(n_layer) * kXcds * M * (2 * kC + (kR + 2) * kHD + kH / kXcds) * sizeof(uint32_t);
    return kDecodeLayersControlBytes + part + local;
}

int launch_decode_layers(const DecodeLayerPointers* layers, int n_layer, const uint16_t* x, const int64_t* tokens,
                         int64_t token_stride, int64_t vocab, uint16_t* out, int M, const float* rope_table, int table_rows, const int* pos, int64_t c_sb, int64_t c_st, int cache_len,
                         float eps, float scale, void* ws, hipStream_t stream) {
    LayersParams p;
    p.layers = layers;
    p.x = x;
    p.tokens = tokens;
    p.token_stride = token_stride;
    p.vocab = vocab;
    p.out = out;
    p.rope_table = rope_table;
    p.pos = pos;
    p.ws = static_cast<unsigned char*>(ws);
    p.c_sb = c_sb;
    p.c_st = c_st;
    p.n_layer = n_layer;
    p.cache_len = cache_len;
    p.table_rows = table_rows;
    p.eps = eps;
    p.scale_log2e = scale * 1.4426950408889634f;
    const dim3 grid(kXcds * kSlots), block(kLayersThreads);
    switch (M) {
        case 1: return enqueue(decode_layers_kernel<1>, grid, block, 0, stream, p);
        case 2: return enqueue(decode_layers_kernel<2>, grid, block, 0, stream, p);
        case 3: return enqueue(decode_layers_kernel<3>, grid, block, 0, stream, p);
        default: return enqueue(decode_layers_kernel<4>, grid, block, 0, stream, p);
    }
}

}  // namespace l3
