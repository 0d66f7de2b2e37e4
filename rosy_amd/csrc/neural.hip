// Material-decoder kernels: latent initialisation, training (forward, backward and Adam), FP16
// export, PSNR evaluation and point decoding.  The decoder itself is defined in neural.h.
//
// Training.  A step draws `batch` samples (u, v) and regresses the decoder onto the plain
// sampler's values there (mean squared error over the 7 channels), then applies one Adam update
// (lr with an optional cosine decay, beta1, beta2, eps) to the latents it touched and to the shared MLP.  Samples are drawn per
// workgroup inside a region of 2^log2R x 2^log2R latent cells of one material, positioned so that
// every bilinear footprint stays inside the region: a workgroup sorts its samples by cell, sums each cell's
// gradient in a register over the cell's samples (in a fixed order, products rounded before they are added) and
// applies Adam to its region itself.  The regions of one step are distinct cells of one partition of every
// grid (the partition shifts by a random offset each step), so no two workgroups touch the same
// latent.  The MLP gradient is reduced per workgroup from per-sample records in LDS and summed over
// workgroups in a fixed order by a second kernel, which also applies Adam to it; after a batch of
// steps a one-thread kernel advances the device-side step counter (each launch of the batch knows how
// many steps it is ahead of it, so a captured graph of steps replays as consecutive steps).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "bin_raster.h"
#include "frame_types.h"
#include "kernels.h"
#include "neural.h"

namespace rsy {
namespace {

constexpr int kMaxR = 32;   // largest region side (explicit mode: the whole grid)
// Per-sample record in LDS for the MLP gradient products, in groups of four words: dL/dhidden 32,
// features 10 and the constant 1 (its products are the bias gradients), dL/dout 7, hidden 32,
// dL/dlatent 8; the sample's two bilinear weights sit in the feature and output groups' spare words.
constexpr int kRec = 92, kRecDh = 0, kRecIn = 32, kRecAx = 43, kRecDo = 44, kRecAy = 51, kRecH = 52, kRecDl = 84;
// The products as 4 x 4 blocks, 16 a wave: dL/dW1 and dL/db1 (8 hidden groups by 3 feature groups),
// dL/dW2 (8 hidden groups by 2 output groups), dL/db2 (the constant's group by 2 output groups).
constexpr uint32_t kGradBlocks1 = 24, kGradBlocks2 = 16, kGradBlocks = kGradBlocks1 + kGradBlocks2 + 2;
constexpr uint32_t kGradWaves = (kGradBlocks + 15) / 16;
static_assert(kGradWaves <= 4, "the sample waves");
constexpr uint32_t kStepThreads = 512;
// A cell with more entries than this in a chunk of an explicit batch is summed by its wave together, in the same order: one
// lane takes 330 cycles an entry, all of its wave's cells beside one another, the wave 110, one cell after the other.  65,536
// samples in one cell: 12 and 8.3 ms (8.5 by atomics).  Training, where a cell has four entries on average, pays more for
// the test than its crowded regions gain (15.4 and 16.5 us a step).
constexpr uint32_t kCrowded = 32;
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline uint64_t mix64(uint64_t z) {  // SplitMix64 finaliser
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__device__ inline float unit24(uint32_t x) { return float(x >> 8) * (1.0f / 16777216.0f); }  // [0, 1)

__device__ inline float mul_rn(float a, float b) {  // rounded by itself: not fused into a later sum
#pragma clang fp contract(off)
    return a * b;
}

// One Adam step of a parameter x with moments m, v; `rate` is the learning rate, bc1 and bc2 the moments' corrections.
__device__ inline void adam_step(float& x, float& m, float& v, float g, const NmTrainLaunch& T, float rate, float bc1,
                                 float bc2) {
    m = fmaf(1.f - T.beta1, g, mul_rn(T.beta1, m));
    v = fmaf(g, mul_rn(1.f - T.beta2, g), mul_rn(T.beta2, v));
    x = x - rate * (m / bc1) / (sqrtf(v / bc2) + T.eps);
}

// Learning-rate factor of step `step`: 0.5 (1 + cos(pi step / decay)) until `decay`, then 0.
__device__ inline float lr_factor(uint32_t step, uint32_t decay) {
    if (decay == 0) return 1.f;
    if (step >= decay) return 0.f;
    return 0.5f * (1.f + cospif(float(step) / float(decay)));
}

__device__ inline float block_sum(float v, float* red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = 0.f;
    if (threadIdx.x == 0)
        for (int w = 0; w < int(blockDim.x >> 6); ++w) s += red[w];
    return s;
}

// Bilinear REPEAT footprint of a sample in a map: the first texel of its two rows, whether the second column
// wraps around (then the rows' first texels are the second column), and the four weights.
struct Taps {
    uint32_t row[2], x;
    bool wraps;
    float w[4];
};
__device__ inline Taps taps_of(const TexGPU& t, float u, float v) {
    const float x = u * float(t.width) - 0.5f, y = v * float(t.height) - 0.5f;
    const float fx = floorf(x), fy = floorf(y), ax = x - fx, ay = y - fy;
    const int x0 = int(fx), y0 = int(fy), w = int(t.width), h = int(t.height);
    const uint32_t xa = uint32_t(wrap_coord(x0, w, 2u));
    const uint32_t ya = uint32_t(wrap_coord(y0, h, 2u)), yb = ya + 1u == t.height ? 0u : ya + 1u;
    return {{ya * t.width, yb * t.width}, xa, xa + 1u == t.width, {(1 - ax) * (1 - ay), ax * (1 - ay), (1 - ax) * ay, ax * ay}};
}

// The training target at (u, v), nm_target's value for the maps a decoded material has (four-channel
// albedo, two-channel normal and metallic-roughness), in two parts: the texels -- the two of a row in
// one load unless the footprint wraps around -- and their mix through the byte tables in LDS (lut[0]
// UNORM, lut[1] sRGB).
struct StepTexels {
    uint32_t a[4], n[4], m[4];
    float wa[4], wn[4], wm[4];
};
template <class T>
__device__ inline void row_pair(const uint8_t* map, const Taps& t, int row, uint32_t& first, uint32_t& second) {
    const T* p = reinterpret_cast<const T*>(map) + t.row[row];
    struct __attribute__((packed)) Pair {
        T a, b;
    };
    if (t.wraps) {
        first = p[t.x];
        second = p[0];
    } else {
        const Pair q = *reinterpret_cast<const Pair*>(p + t.x);
        first = q.a;
        second = q.b;
    }
}
__device__ inline StepTexels step_texels(const uint8_t* texels, const uint8_t* packed, const PackGPU& pk, const TexGPU& ta,
                                         const TexGPU& tn, const TexGPU& tm, float u, float v) {
    if (pk.levels != 0u) {  // the maps as one packed image (a decoded material's samplers repeat)
        const PackTaps q = pack_taps(reinterpret_cast<const uint2*>(packed + pk.offset), int(pk.width), int(pk.height),
                                     2u << kPackWrapS | 2u << kPackWrapT, u, v);
        StepTexels p;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            p.a[k] = q.t[k].x;
            p.n[k] = q.t[k].y & 0xffffu;
            p.m[k] = q.t[k].y >> 16;
            p.wa[k] = p.wn[k] = p.wm[k] = q.w[k];
        }
        return p;
    }
    const Taps a = taps_of(ta, u, v);  // maps of one extent (a uniform test) share their footprint
    Taps n = a, m = a;
    if (tn.width != ta.width || tn.height != ta.height) n = taps_of(tn, u, v);
    if (tm.width != ta.width || tm.height != ta.height) m = taps_of(tm, u, v);
    StepTexels p;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        row_pair<uint32_t>(texels + ta.offset, a, k, p.a[2 * k], p.a[2 * k + 1]);
        row_pair<uint16_t>(texels + tn.offset, n, k, p.n[2 * k], p.n[2 * k + 1]);
        row_pair<uint16_t>(texels + tm.offset, m, k, p.m[2 * k], p.m[2 * k + 1]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        p.wa[k] = a.w[k];
        p.wn[k] = n.w[k];
        p.wm[k] = m.w[k];
    }
    return p;
}
__device__ inline void step_target(const StepTexels& p, const TexGPU& ta, const TexGPU& tn, const TexGPU& tm,
                                   const float (*lut)[256], float (&out)[kNmOut]) {
    const float *la = lut[ta.srgb ? 1 : 0], *ln = lut[tn.srgb ? 1 : 0], *lm = lut[tm.srgb ? 1 : 0];
    const auto mix = [](const float (&w)[4], const uint32_t (&t)[4], uint32_t c, const float* l) {
        const uint32_t s = 8 * c;  // sample_tex's order and roundings
        return fmaf(w[3], l[(t[3] >> s) & 0xffu], fmaf(w[2], l[(t[2] >> s) & 0xffu],
                    fmaf(w[0], l[(t[0] >> s) & 0xffu], mul_rn(w[1], l[(t[1] >> s) & 0xffu]))));
    };
#pragma unroll
    for (uint32_t c = 0; c < 3; ++c) out[c] = mix(p.wa, p.a, c, la);
#pragma unroll
    for (uint32_t c = 0; c < 2; ++c) {
        out[3 + c] = mix(p.wn, p.n, c, ln);
        out[5 + c] = mix(p.wm, p.m, c, lm);
    }
}

// The MLP of a step as outer products: v_mfma_f32_4x4x1 with its A block broadcast adds w[0..3] * x to four
// accumulators of every lane, w the four words of one 4-lane block and x the lane's own value -- so a
// lane keeps its own sample throughout, nothing moves between lanes, the arithmetic is FP32 and the
// weights are 19 registers.  An instruction takes 8 cycles where four multiply-adds take 16.
// Weight word q of a table (block q % 16 of register q / 16) holds rows 4 (q % G) .. +3 of column q / G,
// G groups of four rows; columns run over the bias, then the inputs (forward tables), or the outputs
// of the layer (backward tables).
__device__ inline f32x4 mfma_outer(float w, float x, f32x4 acc, int block) {
#if defined(__HIP_DEVICE_COMPILE__)
    switch (block) {  // the block is an immediate
#define RSY_OUTER(b) case b: return __builtin_amdgcn_mfma_f32_4x4x1f32(w, x, acc, 4, b, 0)
        RSY_OUTER(0); RSY_OUTER(1); RSY_OUTER(2); RSY_OUTER(3); RSY_OUTER(4); RSY_OUTER(5); RSY_OUTER(6); RSY_OUTER(7);
        RSY_OUTER(8); RSY_OUTER(9); RSY_OUTER(10); RSY_OUTER(11); RSY_OUTER(12); RSY_OUTER(13); RSY_OUTER(14);
        default: return __builtin_amdgcn_mfma_f32_4x4x1f32(w, x, acc, 4, 15, 0);
#undef RSY_OUTER
    }
#else
    return acc;
#endif
}
// The tables live in device memory in this form (one coalesced load a register): k_nm_mlp writes a
// parameter's words after its update, k_nm_tables all of them before the first step.
constexpr int kTabF1 = 0, kTabF2 = 6, kTabR2 = 11, kTabR1 = 15;  // [b1 | W1] and [b2 | W2] forward; W2 by hidden unit, W1 by latent channel
static_assert(kTabR1 + 4 == kNmStepTables, "table registers");
// Table words of parameter g (at most two).
struct TableWords {
    uint32_t n, at[2];
};
__host__ __device__ inline uint32_t table_word(int tab, uint32_t groups, uint32_t column, uint32_t row) {
    const uint32_t q = column * groups + row / 4u;
    return (uint32_t(tab) + q / 16u) * 64u + (q % 16u) * 4u + row % 4u;
}
__host__ __device__ inline TableWords table_words(uint32_t g) {
    if (g < uint32_t(kNmB1)) {
        const uint32_t j = g / kNmIn, k = g % kNmIn;
        return {k < uint32_t(kNmCh) ? 2u : 1u, {table_word(kTabF1, 8, k + 1, j), table_word(kTabR1, 2, j, k)}};
    }
    if (g < uint32_t(kNmW2)) return {1u, {table_word(kTabF1, 8, 0, g - kNmB1), 0u}};
    if (g < uint32_t(kNmB2)) {
        const uint32_t c = (g - kNmW2) / kNmHidden, j = (g - kNmW2) % kNmHidden;
        return {2u, {table_word(kTabF2, 2, j + 1, c), table_word(kTabR2, 8, c, j)}};
    }
    return {1u, {table_word(kTabF2, 2, 0, g - kNmB2), 0u}};
}
__device__ inline void write_table(float* tables, const TableWords& w, float x) {
    tables[w.at[0]] = x;
    if (w.n > 1) tables[w.at[1]] = x;
}
// (the words of no parameter stay the zeros the buffer was allocated with)
__global__ __launch_bounds__(256) void k_nm_tables(const float* mlp, float* tables) {
    const uint32_t g = blockIdx.x * 256 + threadIdx.x;
    if (g < uint32_t(kNmParams)) write_table(tables, table_words(g), mlp[g]);
}

// One training step's samples: a workgroup per region; a thread of its first four waves per sample, the
// other four hold the region's cells.
//
// A step has 65,536 samples by default: one sample wave on each of the chip's 1,024 SIMDs, so the kernel's
// time is the length of one wave's chain: the step counter, the slot's map records, the texels (each
// launch starts with a cold L2: 2,000 cycles a hop), the MLP, its gradient.
// - Loads that depend on nothing else go out together at the start; the cell waves load the region's Adam
//   state, whose latents the samples read from LDS.
// - A sample's texels come from its material's packed image: four loads on 1.6 lines instead of six loads on
//   six lines (4.3 us a step less: the texel pages and lines of 65,536 samples), which maps that cannot be packed keep.
// - The MLP runs in registers on the matrix cores (its weights were read from LDS, one wait per hidden unit).
// - Its gradient, a product over the samples, is one matrix instruction per sample and wave from
//   records in LDS: 256 multiply-adds in sample order for every parameter, as the scalar loops had it
//   (three dot products of 256 LDS pairs a thread, 20,000 cycles), 29 cycles apart.
// - Latent gradients were 32 LDS float atomics a sample (20,000 cycles): the samples are sorted by cell
//   while their texels are on the way, and the cell waves sum them and apply Adam beside the MLP gradient.
//   A sample's place in its cell follows the samples' order, not the arrival of threads, and a product is rounded
//   before it is added, as an atomic's operand is: Adam divides by the root of a second moment that may be as small as
//   the rounding, so other last bits become other steps (two runs by atomics are 4e-5 apart after 512 steps).  The
//   sets that give the places take 1 us of the step.
// 65,536 samples of 16 materials: 47 us before, 15.4 us; the MLP's update 6.2 and 5.3 us.
template <bool kExplicit>
__global__ __launch_bounds__(kStepThreads) void k_nm_step(NmTrainLaunch T) {
    constexpr uint32_t kMaxCells = kMaxR * kMaxR, kCellsPerThread = kMaxCells / 256;
    __shared__ __align__(16) float rec_s[256 * kRec];
    __shared__ __align__(16) float4 lat_s[2 * kMaxCells];        // the region's latents, 8 a cell
    __shared__ uint32_t count_s[kMaxCells], first_s[kMaxCells];  // samples per base cell and their first entry in order_s
    __shared__ uint16_t order_s[256];                            // the chunk's samples by base cell
    __shared__ uint32_t scan_s[kStepThreads / 64];
    __shared__ float sum_s[kNmParamsPad];
    __shared__ float lut[2][256];
    __shared__ float red_s[kStepThreads / 64];
    // waves 0..3 take the samples, waves 4..7 the region's cells
    const uint32_t lane = threadIdx.x & 63u, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
    const bool sampler = wave < 4;
    const uint32_t tid = threadIdx.x & 255u;
    const uint32_t step = kExplicit ? 0u : *T.step + T.step_ahead;
    const uint32_t L = T.L, Lm = L - 1;
    const float inv_L = 1.f / float(L);  // exact: a power of two
    float W[kNmStepTables] = {};
    if (sampler)
#pragma unroll
        for (int v = 0; v < kNmStepTables; ++v) W[v] = T.tables[v * 64 + lane];

    uint32_t slot, rx, ry, R, log2R;
    if (kExplicit) {
        slot = blockIdx.x;
        rx = ry = 0;
        R = L;
        log2R = T.log2L;
    } else {
        log2R = T.log2R;
        R = 1u << log2R;
        const uint32_t log2rx = T.log2L - log2R;
        const uint32_t rpm = 1u << (2 * log2rx);  // regions per grid
        const uint64_t n_regions = uint64_t(T.n_slots) * rpm;
        const uint64_t r = (uint64_t(step) * T.n_wg + blockIdx.x) % n_regions;
        slot = uint32_t(r % T.n_slots);
        const uint32_t reg = (uint32_t(r / T.n_slots) * 2654435761u) & (rpm - 1);  // odd multiplier: a bijection
        const uint64_t hs = mix64(T.seed ^ mix64(0x5bd1e995ull + step));
        const uint32_t ox = uint32_t(hs) & (R - 1), oy = uint32_t(hs >> 32) & (R - 1);
        rx = (reg & ((1u << log2rx) - 1)) * R + ox;
        ry = (reg >> log2rx) * R + oy;
    }
    const uint32_t cells = R * R;
    const size_t grid_base = size_t(slot) * L * L;
    auto cell_of = [&](uint32_t cx, uint32_t cy) { return grid_base + size_t((ry + cy) & Lm) * L + ((rx + cx) & Lm); };
    TexGPU ta{}, tn{}, tm{};
    PackGPU pk{};
    float4 adam[6] = {};  // a cell wave: the Adam state of the thread's first cell, and the step's factors
    float bc1 = 1.f, bc2 = 1.f, lr = 0.f;
    if (sampler) {
        ta = T.maps[3 * slot];
        tn = T.maps[3 * slot + 1];
        tm = T.maps[3 * slot + 2];
        pk = T.packs[slot];
    } else {
        const float srgb = T.srgb_lut[tid];
        if (!kExplicit && tid < cells) {
            const size_t g = 2 * cell_of(tid & (R - 1), tid >> log2R);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                adam[k] = reinterpret_cast<const float4*>(T.lat)[g + k];
                adam[2 + k] = reinterpret_cast<const float4*>(T.lat_m)[g + k];
                adam[4 + k] = reinterpret_cast<const float4*>(T.lat_v)[g + k];
            }
        }
        for (uint32_t i = tid; i < cells; i += 256) {
            if (!kExplicit && i < 256) {
                lat_s[2 * i] = adam[0];
                lat_s[2 * i + 1] = adam[1];
            } else {
                const size_t g = 2 * cell_of(i & (R - 1), i >> log2R);
                lat_s[2 * i] = reinterpret_cast<const float4*>(T.lat)[g];
                lat_s[2 * i + 1] = reinterpret_cast<const float4*>(T.lat)[g + 1];
            }
        }
        lut[0][tid] = float(tid) * (1.0f / 255.0f);
        lut[1][tid] = srgb;
        const float t = float(step + 1);
        bc1 = 1.f - powf(T.beta1, t);
        bc2 = 1.f - powf(T.beta2, t);
        lr = T.lr_lat * lr_factor(step, T.decay_steps);
    }

    uint32_t n_samples, s_base = 0;
    if (kExplicit) {
        s_base = T.ex_offsets[slot];
        n_samples = T.ex_offsets[slot + 1] - s_base;
    } else {
        n_samples = T.spw;
    }
    const uint64_t skey = mix64(T.seed + 0x632BE59BD9B4E019ull * (uint64_t(step) + 1)) + (uint64_t(blockIdx.x) << 32);
    float* const rec = rec_s + tid * kRec;
    // the lane's block of the gradient products: its row operand and column operand in a record
    const uint32_t blk = wave * 16u + (lane >> 2), blk2 = blk - kGradBlocks1;
    const bool first_layer = blk < kGradBlocks1, bias2 = blk >= kGradBlocks1 + kGradBlocks2;
    const uint32_t row_at = (first_layer ? kRecDh + 4u * (blk / 3u) : bias2 ? kRecIn + 8u : kRecH + 4u * (blk2 / 2u)) + (lane & 3u);
    const uint32_t col_at = (first_layer ? kRecIn + 4u * (blk % 3u) : kRecDo + 4u * (blk2 % 2u)) + (lane & 3u);
    f32x4 grad = {};                          // of the lane's block
    float grad_lat[kCellsPerThread][kNmCh] = {};  // of the thread's cells tid, tid + 256, ...
    float loss = 0.f;
    for (uint32_t base = 0; base < n_samples; base += 256) {
        const uint32_t q = base + tid;
        const bool live = sampler && q < n_samples;
        float tgt[kNmOut] = {}, ax = 0.f, ay = 0.f;
        uint32_t i0 = 0, i1 = 0, j0 = 0, j1 = 0;
        StepTexels px{};
        if (live) {
            float u, v;
            if (kExplicit) {
                u = T.ex_uv[2 * size_t(s_base + q)];
                v = T.ex_uv[2 * size_t(s_base + q) + 1];
                const float x = u * float(L) - 0.5f, y = v * float(L) - 0.5f;
                const float fx = floorf(x), fy = floorf(y);
                ax = x - fx;
                ay = y - fy;
                i0 = uint32_t(int(fx)) & Lm;
                j0 = uint32_t(int(fy)) & Lm;
                i1 = (i0 + 1) & Lm;
                j1 = (j0 + 1) & Lm;
            } else {
                const uint64_t hh = mix64(skey + q);
                const float sx = unit24(uint32_t(hh)), sy = unit24(uint32_t(hh >> 32)), span = float(R - 1);
                const float xl = mul_rn(sx, span), yl = mul_rn(sy, span);
                i0 = min(uint32_t(xl), R - 2);
                j0 = min(uint32_t(yl), R - 2);
                ax = xl - float(i0);
                ay = yl - float(j0);
                u = (fmaf(sx, span, float(rx)) + 0.5f) * inv_L;
                v = (fmaf(sy, span, float(ry)) + 0.5f) * inv_L;
                i1 = i0 + 1;
                j1 = j0 + 1;
            }
            if (kExplicit) {
#pragma unroll
                for (int c = 0; c < kNmOut; ++c) tgt[c] = T.ex_target[kNmOut * size_t(s_base + q) + c];
            } else {
                px = step_texels(T.texels, T.packed, pk, ta, tn, tm, u, v);
            }
        }
        // the chunk's samples sorted by base cell, in their order within a cell, while their texels and cells are on
        // the way: a cell's set of samples is 256 bits (in the records' space, which is free until they are written),
        // a sample's place in the cell its bits below the sample's own
        uint4* const set_s = reinterpret_cast<uint4*>(rec_s);
        for (uint32_t i = threadIdx.x; i < 2 * cells; i += kStepThreads) set_s[i] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();  // sets cleared, tables written
        const uint32_t bin = j0 * R + i0;
        if (live) atomicOr(reinterpret_cast<uint32_t*>(set_s + 2 * bin) + (tid >> 5), 1u << (tid & 31u));
        __syncthreads();
        uint32_t rank = 0;
        if (live) {
            const uint4 s0 = set_s[2 * bin], s1 = set_s[2 * bin + 1];
            const uint32_t w[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) rank += __popc(k < (tid >> 5) ? w[k] : k == (tid >> 5) ? w[k] & ((1u << (tid & 31u)) - 1u) : 0u);
        }
        {
            uint32_t n[kCellsPerThread] = {}, mine = 0, total;
#pragma unroll
            for (uint32_t k = 0; k < kCellsPerThread; ++k) {
                const uint32_t c = tid * kCellsPerThread + k;
                if (!sampler && c < cells) {
                    const uint4 s0 = set_s[2 * c], s1 = set_s[2 * c + 1];
                    n[k] = __popc(s0.x) + __popc(s0.y) + __popc(s0.z) + __popc(s0.w) + __popc(s1.x) + __popc(s1.y) + __popc(s1.z) + __popc(s1.w);
                    count_s[c] = n[k];
                }
                mine += n[k];
            }
            uint32_t at = block_exclusive_scan(mine, scan_s, total);
#pragma unroll
            for (uint32_t k = 0; k < kCellsPerThread; ++k) {
                const uint32_t c = tid * kCellsPerThread + k;
                if (!sampler && c < cells) first_s[c] = at;
                at += n[k];
            }
        }
        __syncthreads();
        if (sampler) {
            if (live) order_s[first_s[bin] + rank] = uint16_t(tid);
            float in[kNmIn] = {};
            if (live) {
                const float w00 = (1.f - ax) * (1.f - ay), w10 = ax * (1.f - ay), w01 = (1.f - ax) * ay, w11 = ax * ay;
                const float4 *q00 = lat_s + 2 * (j0 * R + i0), *q10 = lat_s + 2 * (j0 * R + i1);
                const float4 *q01 = lat_s + 2 * (j1 * R + i0), *q11 = lat_s + 2 * (j1 * R + i1);
                const float4 c00[2] = {q00[0], q00[1]}, c10[2] = {q10[0], q10[1]};
                const float4 c01[2] = {q01[0], q01[1]}, c11[2] = {q11[0], q11[1]};
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    in[4 * k + 0] = w00 * c00[k].x + w10 * c10[k].x + w01 * c01[k].x + w11 * c11[k].x;
                    in[4 * k + 1] = w00 * c00[k].y + w10 * c10[k].y + w01 * c01[k].y + w11 * c11[k].y;
                    in[4 * k + 2] = w00 * c00[k].z + w10 * c10[k].z + w01 * c01[k].z + w11 * c11[k].z;
                    in[4 * k + 3] = w00 * c00[k].w + w10 * c10[k].w + w01 * c01[k].w + w11 * c11[k].w;
                }
                in[8] = 1.f - fabsf(2.f * ax - 1.f);
                in[9] = 1.f - fabsf(2.f * ay - 1.f);
                if (!kExplicit) step_target(px, ta, tn, tm, lut, tgt);
            }
            // forward and backward in every lane (a lane without a sample has zero features and zero dL/dout)
            f32x4 acc[8], o2[2] = {}, dz[8], din[2] = {};
#pragma unroll
            for (int g = 0; g < 8; ++g) acc[g] = mfma_outer(W[kTabF1 + g / 16], 1.f, f32x4{}, g % 16);
#pragma unroll
            for (int k = 0; k < kNmIn; ++k)
#pragma unroll
                for (int g = 0; g < 8; ++g) acc[g] = mfma_outer(W[kTabF1 + (8 * k + 8 + g) / 16], in[k], acc[g], (8 * k + 8 + g) % 16);
            float h[kNmHidden], dh[kNmHidden], dout[kNmOut];
#pragma unroll
            for (int j = 0; j < kNmHidden; ++j) h[j] = fmaxf(acc[j / 4][j % 4], 0.f);
#pragma unroll
            for (int g = 0; g < 2; ++g) o2[g] = mfma_outer(W[kTabF2], 1.f, f32x4{}, g);
#pragma unroll
            for (int j = 0; j < kNmHidden; ++j)
#pragma unroll
                for (int g = 0; g < 2; ++g) o2[g] = mfma_outer(W[kTabF2 + (2 * j + 2 + g) / 16], h[j], o2[g], (2 * j + 2 + g) % 16);
#pragma unroll
            for (int c = 0; c < kNmOut; ++c) {
                const float d = live ? o2[c / 4][c % 4] - tgt[c] : 0.f;
                loss += d * d;
                dout[c] = 2.f * d * T.inv_norm;
            }
            // backward: dL/dhidden (ReLU mask), dL/dfeatures for the 8 latent channels
#pragma unroll
            for (int g = 0; g < 8; ++g) dz[g] = mfma_outer(W[kTabR2], dout[0], f32x4{}, g);
#pragma unroll
            for (int c = 1; c < kNmOut; ++c)
#pragma unroll
                for (int g = 0; g < 8; ++g) dz[g] = mfma_outer(W[kTabR2 + (8 * c + g) / 16], dout[c], dz[g], (8 * c + g) % 16);
#pragma unroll
            for (int j = 0; j < kNmHidden; ++j) dh[j] = h[j] > 0.f ? dz[j / 4][j % 4] : 0.f;
#pragma unroll
            for (int j = 0; j < kNmHidden; ++j)
#pragma unroll
                for (int g = 0; g < 2; ++g) din[g] = mfma_outer(W[kTabR1 + (2 * j + g) / 16], dh[j], din[g], (2 * j + g) % 16);
            // the sample's record (zeros past the last sample: no contribution)
#pragma unroll
            for (int k = 0; k < kNmHidden; k += 4) {
                *reinterpret_cast<float4*>(rec + kRecDh + k) = make_float4(dh[k], dh[k + 1], dh[k + 2], dh[k + 3]);
                *reinterpret_cast<float4*>(rec + kRecH + k) = make_float4(h[k], h[k + 1], h[k + 2], h[k + 3]);
            }
            *reinterpret_cast<float4*>(rec + kRecIn) = make_float4(in[0], in[1], in[2], in[3]);
            *reinterpret_cast<float4*>(rec + kRecIn + 4) = make_float4(in[4], in[5], in[6], in[7]);
            *reinterpret_cast<float4*>(rec + kRecIn + 8) = make_float4(in[8], in[9], 1.f, ax);
            *reinterpret_cast<float4*>(rec + kRecDo) = make_float4(dout[0], dout[1], dout[2], dout[3]);
            *reinterpret_cast<float4*>(rec + kRecDo + 4) = make_float4(dout[4], dout[5], dout[6], ay);
            *reinterpret_cast<f32x4*>(rec + kRecDl) = din[0];
            *reinterpret_cast<f32x4*>(rec + kRecDl + 4) = din[1];
        }
        __syncthreads();
        // each wave its sixteen blocks over all records, one sample an instruction: every gradient is the
        // multiply-add chain over the samples in their order, whatever the wave that runs it.  A batch of
        // operands is read while the last one goes through the chain.
        if (wave < kGradWaves) {
            constexpr uint32_t kBatch = 16;
            const float* const pr = rec_s + min(row_at, uint32_t(kRec - 1));
            const float* const pc = rec_s + min(col_at, uint32_t(kRec - 1));
            f32x4 s = {};
            const uint32_t cnt = min(256u, n_samples - base);  // records from cnt on are zeros
            float a[kBatch], b[kBatch];
#pragma unroll
            for (uint32_t k = 0; k < kBatch; ++k) {
                a[k] = pr[k * kRec];
                b[k] = pc[k * kRec];
            }
            for (uint32_t r = 0; r < cnt; r += kBatch) {
                float na[kBatch], nb[kBatch];
                const uint32_t next = min(r + kBatch, 256u - kBatch);
#pragma unroll
                for (uint32_t k = 0; k < kBatch; ++k) {
                    na[k] = pr[(next + k) * kRec];
                    nb[k] = pc[(next + k) * kRec];
                }
#pragma unroll
                for (uint32_t k = 0; k < kBatch; ++k) s = __builtin_amdgcn_mfma_f32_4x4x1f32(a[k], b[k], s, 0, 0, 0);
#pragma unroll
                for (uint32_t k = 0; k < kBatch; ++k) {
                    a[k] = na[k];
                    b[k] = nb[k];
                }
            }
            grad += s;
        }
        // meanwhile the cell waves gather: a cell is a corner of four base cells' samples (a base cell in the last
        // column or row has no samples in a region, and wraps around in a whole grid); the four lists are
        // walked as one, the next sample's place read ahead
        if (!sampler) {
#pragma unroll
            for (uint32_t k = 0; k < kCellsPerThread; ++k) {
                if ((kExplicit ? 0u : tid) + 256u * k >= cells) break;  // (an explicit batch's waves stay together)
                const uint32_t cell = kExplicit ? min(tid + 256u * k, cells - 1u) : tid + 256u * k;
                const uint32_t cx = cell & (R - 1), cy = cell >> log2R;
                uint32_t end[4], at[4], n = 0;
#pragma unroll
                for (uint32_t c = 0; c < 4; ++c) {
                    const uint32_t from = ((cy - (c >> 1)) & (R - 1)) * R + ((cx - (c & 1u)) & (R - 1));
                    at[c] = first_s[from] - n;  // entry i of the joint list: at[c] + i for i in [end[c - 1], end[c])
                    n += count_s[from];
                    end[c] = n;
                }
                unsigned long long owners = 0ull;
                if constexpr (kExplicit) {
                    if (tid + 256u * k >= cells) n = 0;
                    const bool crowded = n > kCrowded;
                    owners = __builtin_amdgcn_ballot_w64(crowded);
                    if (crowded) n = 0;
                }
                const auto place = [&](uint32_t i) {
                    const uint32_t a = i < end[0] ? at[0] : i < end[1] ? at[1] : i < end[2] ? at[2] : at[3];
                    return uint32_t(order_s[min(a + i, 255u)]) * kRec;
                };
                uint32_t o = n ? place(0) : 0u;
                for (uint32_t i = 0; i < n; ++i) {
                    const float* r = rec_s + o;
                    const float x = r[kRecAx], y = r[kRecAy];
                    const f32x4 d0 = *reinterpret_cast<const f32x4*>(r + kRecDl), d1 = *reinterpret_cast<const f32x4*>(r + kRecDl + 4);
                    o = place(i + 1);
                    const bool right = (i >= end[0] && i < end[1]) || i >= end[2], low = i >= end[1];
                    const float w = (right ? x : 1.f - x) * (low ? y : 1.f - y);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        grad_lat[k][c] += mul_rn(w, d0[c]);
                        grad_lat[k][4 + c] += mul_rn(w, d1[c]);
                    }
                }
                // a crowded cell of an explicit batch: its wave takes eight entries at a time, a lane one channel of one of them, and adds the
                // eight products of a channel in the entries' order
                for (; kExplicit && owners != 0ull; owners &= owners - 1ull) {  // uniform
                    const int owner = __builtin_ctzll(owners);
                    uint32_t oe[4], oa[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        oe[c] = uint32_t(__builtin_amdgcn_readlane(int(end[c]), owner));
                        oa[c] = uint32_t(__builtin_amdgcn_readlane(int(at[c]), owner));
                    }
                    const uint32_t channel = lane & 7u;
                    float sum = 0.f;
#pragma unroll
                    for (uint32_t c = 0; c < kNmCh; ++c) {
                        const float v = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(grad_lat[k][c]), owner));
                        if (channel == c) sum = v;
                    }
                    for (uint32_t i = 0; i < oe[3]; i += 8) {
                        const uint32_t e = i + (lane >> 3);
                        const uint32_t a = e < oe[0] ? oa[0] : e < oe[1] ? oa[1] : e < oe[2] ? oa[2] : oa[3];
                        const float* r = rec_s + uint32_t(order_s[min(a + e, 255u)] & 255u) * kRec;
                        const bool right = (e >= oe[0] && e < oe[1]) || e >= oe[2], low = e >= oe[1];
                        const float x = r[kRecAx], y = r[kRecAy];
                        const float product = mul_rn((right ? x : 1.f - x) * (low ? y : 1.f - y), r[kRecDl + channel]);
#pragma unroll
                        for (uint32_t q = 0; q < 8; ++q) {
                            const float v = __shfl(product, int(8u * q + channel));
                            if (i + q < oe[3]) sum += v;
                        }
                    }
#pragma unroll
                    for (uint32_t c = 0; c < kNmCh; ++c) {
                        const float v = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sum), int(c)));
                        if (lane == uint32_t(owner)) grad_lat[k][c] = v;
                    }
                }
            }
        }
        __syncthreads();
    }
    // latents of the region: gradient out (explicit mode) or Adam
    if (!sampler) {
#pragma unroll
        for (uint32_t k = 0; k < kCellsPerThread; ++k) {
            const uint32_t cell = tid + 256u * k;
            if (cell >= cells) break;
            const size_t g = 2 * cell_of(cell & (R - 1), cell >> log2R);
            if (!kExplicit && k > 0)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    adam[i] = reinterpret_cast<const float4*>(T.lat)[g + i];
                    adam[2 + i] = reinterpret_cast<const float4*>(T.lat_m)[g + i];
                    adam[4 + i] = reinterpret_cast<const float4*>(T.lat_v)[g + i];
                }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float* gr = grad_lat[k] + 4 * i;
                if (kExplicit) {
                    reinterpret_cast<float4*>(T.ex_grad_lat)[g + i] = make_float4(gr[0], gr[1], gr[2], gr[3]);
                } else {
                    float4 &x = adam[i], &m = adam[2 + i], &v = adam[4 + i];
                    adam_step(x.x, m.x, v.x, gr[0], T, lr, bc1, bc2);
                    adam_step(x.y, m.y, v.y, gr[1], T, lr, bc1, bc2);
                    adam_step(x.z, m.z, v.z, gr[2], T, lr, bc1, bc2);
                    adam_step(x.w, m.w, v.w, gr[3], T, lr, bc1, bc2);
                    reinterpret_cast<float4*>(T.lat)[g + i] = x;
                    reinterpret_cast<float4*>(T.lat_m)[g + i] = m;
                    reinterpret_cast<float4*>(T.lat_v)[g + i] = v;
                }
            }
        }
    }
    // the workgroup's sums: a lane holds rows 0..3 of its block's column lane % 4
    if (sampler && blk < kGradBlocks) {
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t col = 4u * (first_layer ? blk % 3u : blk2 % 2u) + (lane & 3u);
            const uint32_t j = 4u * (first_layer ? blk / 3u : blk2 / 2u) + i;
            if (first_layer) {
                if (col < uint32_t(kNmIn)) sum_s[kNmW1 + j * kNmIn + col] = grad[i];
                else if (col == uint32_t(kNmIn)) sum_s[kNmB1 + j] = grad[i];
            } else if (col < uint32_t(kNmOut)) {
                if (!bias2) sum_s[kNmW2 + col * kNmHidden + j] = grad[i];
                else if (i == uint32_t(kNmIn) - 8u) sum_s[kNmB2 + col] = grad[i];
            }
        }
    }
    const float loss_sum = block_sum(loss, red_s);  // synchronises
    if (threadIdx.x == 0) sum_s[kNmParams] = loss_sum;
    __syncthreads();
    // workgroup-major: partial[workgroup * 584 + g], the loss last
    for (uint32_t g = threadIdx.x; g < uint32_t(kNmParamsPad); g += kStepThreads) T.partial[size_t(blockIdx.x) * kNmParamsPad + g] = sum_s[g];
}

// The MLP's update: a block per 64 parameters (one a lane), its 16 waves summing the workgroups'
// partials -- coalesced rows, a wave's rows in flight together -- in a fixed order: 64 strided sums (the
// workgroups i, i + 64, ... of sum i), then those pairwise, i with i + 32, then + 16, + 8, ... -- then Adam (or, in explicit
// mode, the summed gradient) and the step's loss.  6.2 us as one wave per parameter over a
// parameter-major table, 5.3 us.
constexpr uint32_t kMlpWaves = 16;
template <bool kExplicit>
__global__ __launch_bounds__(64 * kMlpWaves) void k_nm_mlp(NmTrainLaunch T) {
    __shared__ float sums[kMlpWaves][64];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, g = blockIdx.x * 64 + lane;
    const bool live = g < uint32_t(kNmParamsPad);
    const uint32_t step = kExplicit ? 0u : *T.step + T.step_ahead;
    float m = 0.f, v = 0.f, x = 0.f;
    const TableWords words = table_words(min(g, uint32_t(kNmParams - 1)));
    const bool update = !kExplicit && wave == 0 && g < uint32_t(kNmParams);
    if (update) {
        m = T.mlp_m[g];
        v = T.mlp_v[g];
        x = T.mlp[g];
    }
    float s4[4] = {};  // sums wave, wave + 16, wave + 32, wave + 48
    if (live)
        for (uint32_t b = wave; b < T.n_wg; b += 256) {
            float p[4][4];
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) {
                    const uint32_t wg = b + 64 * k + 16 * i;
                    p[k][i] = wg < T.n_wg ? T.partial[size_t(wg) * kNmParamsPad + g] : 0.f;
                }
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) s4[i] += p[k][i];
        }
    sums[wave][lane] = (s4[0] + s4[2]) + (s4[1] + s4[3]);
#pragma unroll
    for (uint32_t o = kMlpWaves / 2; o > 0; o >>= 1) {
        __syncthreads();
        if (wave < o) sums[wave][lane] += sums[wave + o][lane];
    }
    if (wave != 0 || !live) return;
    const float s = sums[0][lane];
    if (kExplicit) {
        T.ex_grad_mlp[g] = s;
    } else if (update) {
        const float t = float(step + 1);
        const float bc1 = 1.f - powf(T.beta1, t), bc2 = 1.f - powf(T.beta2, t);
        const float lr = T.lr_mlp * lr_factor(step, T.decay_steps);
        adam_step(x, m, v, s, T, lr, bc1, bc2);
        T.mlp_m[g] = m;
        T.mlp_v[g] = v;
        T.mlp[g] = x;
        write_table(T.tables, words, x);
    } else if (T.loss_out && step >= T.loss_base && step - T.loss_base < T.loss_cap) {
        T.loss_out[step - T.loss_base] = s * T.inv_norm;  // mean squared error of the step
    }
}

// Advances the device step counter by a batch of steps, once their readers have finished.
__global__ void k_nm_advance(uint32_t* step, uint32_t steps) {
    if (threadIdx.x == 0) *step += steps;
}

__global__ __launch_bounds__(256) void k_nm_init(NmInitLaunch I) {
    const uint64_t cells = uint64_t(I.n_slots) * I.L * I.L;
    const NmSlot* slots = static_cast<const NmSlot*>(I.slots);
    for (uint64_t cell = uint64_t(blockIdx.x) * 256 + threadIdx.x; cell < cells; cell += uint64_t(gridDim.x) * 256) {
        float* o = I.lat + cell * kNmCh;
        if (I.random) {
            const uint64_t h = mix64(I.seed ^ mix64(cell));
            const uint64_t h2 = mix64(h);
            const uint32_t r[8] = {uint32_t(h), uint32_t(h >> 32), uint32_t(h2), uint32_t(h2 >> 32),
                                   uint32_t(mix64(h2)), uint32_t(mix64(h2) >> 32), uint32_t(mix64(h2 + 1)),
                                   uint32_t(mix64(h2 + 1) >> 32)};
            for (int c = 0; c < kNmCh; ++c) o[c] = 0.2f * unit24(r[c]) - 0.1f;
        } else {
            const uint32_t slot = uint32_t(cell / (uint64_t(I.L) * I.L));
            const uint32_t local = uint32_t(cell % (uint64_t(I.L) * I.L));
            const float u = (float(local % I.L) + 0.5f) / float(I.L), v = (float(local / I.L) + 0.5f) / float(I.L);
            float tgt[kNmOut];
            nm_target(I.texels, I.textures, slots[slot], u, v, I.srgb_lut, tgt);
            for (int c = 0; c < kNmOut; ++c) o[c] = tgt[c];
            o[7] = 0.f;
        }
    }
}

// FP32 latents to halves; the last block's first wave writes the MLP's operand form instead (a launch
// of its own took 8 us beside the latents' 17).
__device__ void export_weights(const float* p, NmWeights* W, uint32_t fp8);

__global__ __launch_bounds__(256) void k_nm_export(const float* lat, uint4* lat16, uint64_t cells, const float* mlp,
                                                   NmWeights* W, uint32_t fp8) {
    if (blockIdx.x + 1 == gridDim.x) {
        if (threadIdx.x < 64) export_weights(mlp, W, fp8);
        return;
    }
    const uint32_t blocks = gridDim.x - 1;
    for (uint64_t cell = uint64_t(blockIdx.x) * 256 + threadIdx.x; cell < cells; cell += uint64_t(blocks) * 256) {
        const float4 a = reinterpret_cast<const float4*>(lat)[2 * cell];
        const float4 b = reinterpret_cast<const float4*>(lat)[2 * cell + 1];
        const h2 p0 = h2{_Float16(a.x), _Float16(a.y)}, p1 = h2{_Float16(a.z), _Float16(a.w)};
        const h2 p2 = h2{_Float16(b.x), _Float16(b.y)}, p3 = h2{_Float16(b.z), _Float16(b.w)};
        lat16[cell] = make_uint4(__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1),
                                 __builtin_bit_cast(uint32_t, p2), __builtin_bit_cast(uint32_t, p3));
    }
}

// Two neighbouring cells of a latent grid interpolated.
__device__ inline void nm_row(uint4 a, uint4 b, float t, float (&out)[kNmCh]) {
    const uint32_t p[4] = {a.x, a.y, a.z, a.w}, q[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const h2 x = __builtin_bit_cast(h2, p[k]), y = __builtin_bit_cast(h2, q[k]);
        out[2 * k] = (1.f - t) * float(x[0]) + t * float(y[0]);
        out[2 * k + 1] = (1.f - t) * float(x[1]) + t * float(y[1]);
    }
}

// Squared error of the decoder over every texel centre of one slot's albedo map, a block per tile of
// kNmEvalW x kNmEvalH texels: lane = column, a wave walks kNmEvalH / 4 rows.
//
// kTexel: the slot's three maps share one extent, so that the plain sampler at a texel centre is the
// texel itself (bilinear weights 1, 0, 0, 0: in FP32 exactly so for extents that are powers of two, for others within
// the rounding of the coordinates, which reading the texel leaves out): three loads and seven table reads, against twelve loads
// with addressing and format branches.  Slots whose maps differ in size sample bilinearly
// (kTexel = false); each launch passes over the other kind's slots.
//
// Bound by VALU issue: 64 texels take about 230 instructions of 4 cycles (half splits, clamps, error) next to 12
// matrix instructions of 32; texels and latents are 12 bytes a texel.  The rows of a wave share the
// weights, the column's addresses and most cell rows.  32 materials of 1024^2 texels with 256^2 latents: 850 us
// with 256-texel blocks, four cells and twelve texels per texel, 350 us this way (49 us of
// memory time; 16 rows a wave: 344 us, at 3 waves a SIMD instead of 4).
template <bool kTexel>
__global__ __launch_bounds__(256) void k_nm_eval(NmEvalLaunch E) {
    __shared__ float red_s[4];
    __shared__ float lut[2][256];  // stored byte -> value: UNORM, sRGB
    lut[0][threadIdx.x] = float(threadIdx.x) * (1.0f / 255.0f);
    lut[1][threadIdx.x] = E.srgb_lut[threadIdx.x];
    __syncthreads();
    for (uint32_t slot = blockIdx.y; slot < E.n_slots; slot += gridDim.y) {
        const NmSlot S = static_cast<const NmSlot*>(E.slots)[slot];
        const TexGPU ta = E.textures[S.albedo], tn = E.textures[S.normal], tm = E.textures[S.mr];
        const bool same = tn.width == ta.width && tn.height == ta.height && tm.width == ta.width && tm.height == ta.height;
        const uint32_t tiles_x = (ta.width + kNmEvalW - 1) / kNmEvalW, tiles_y = (ta.height + kNmEvalH - 1) / kNmEvalH;
        if (same != kTexel || blockIdx.x >= tiles_x * tiles_y) continue;  // uniform
        const uint32_t x = (blockIdx.x % tiles_x) * kNmEvalW + (threadIdx.x & 63u);
        const uint32_t y0 = (blockIdx.x / tiles_x) * kNmEvalH +
                            uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6))) * (kNmEvalH / 4);
        const uint32_t xc = min(x, ta.width - 1);
        const float u = (float(xc) + 0.5f) / float(ta.width);
        const uint32_t* albedo = reinterpret_cast<const uint32_t*>(E.texels + ta.offset) + xc;
        const uint16_t* normal = reinterpret_cast<const uint16_t*>(E.texels + tn.offset) + xc;
        const uint16_t* mr = reinterpret_cast<const uint16_t*>(E.texels + tm.offset) + xc;
        const float *la = lut[ta.srgb ? 1 : 0], *ln = lut[tn.srgb ? 1 : 0], *lm = lut[tm.srgb ? 1 : 0];
        const uint4* grid = E.lat16 + size_t(slot) * E.L * E.L;
        // the column's two cell columns and weight; the two cell rows around a texel row, interpolated
        // along x and kept while the next texel row lies between the same ones (rows are uniform over the wave)
        const float gx = u * float(E.L) - 0.5f, fx = floorf(gx), ax = gx - fx;
        const uint32_t mask = E.L - 1, cx0 = uint32_t(int(fx)) & mask, cx1 = (cx0 + 1) & mask;
        float lower[kNmCh], slope[kNmCh], upper[kNmCh];  // row cy, row cy + 1 less row cy, row cy + 1
        uint32_t at = 0xffffffffu;                       // the row in `lower` (none yet)
        float err = 0.f;
        for (uint32_t j = 0; j < kNmEvalH / 4; ++j) {
            const uint32_t yc = min(y0 + j, ta.height - 1);
            const float v = (float(yc) + 0.5f) / float(ta.height);
            const size_t row = size_t(yc) * ta.width;
            uint32_t pa = 0, pn = 0, pm = 0;
            if constexpr (kTexel) {
                pa = albedo[row];
                pn = normal[row];
                pm = mr[row];
            }
            const float gy = v * float(E.L) - 0.5f, fy = floorf(gy), ay = gy - fy;
            const uint32_t cy = uint32_t(int(fy)) & mask;
            if (cy != at) {
                if (at != 0xffffffffu && cy == ((at + 1) & mask)) {
#pragma unroll
                    for (int c = 0; c < kNmCh; ++c) lower[c] = upper[c];
                } else {
                    nm_row(grid[cy * E.L + cx0], grid[cy * E.L + cx1], ax, lower);
                }
                const uint32_t cy1 = (cy + 1) & mask;
                nm_row(grid[cy1 * E.L + cx0], grid[cy1 * E.L + cx1], ax, upper);
#pragma unroll
                for (int c = 0; c < kNmCh; ++c) slope[c] = upper[c] - lower[c];
                at = cy;
            }
            float f[kNmFeat];
#pragma unroll
            for (int c = 0; c < kNmCh; ++c) f[c] = fmaf(ay, slope[c], lower[c]);
            f[8] = 1.f - fabsf(2.f * ax - 1.f);
            f[9] = 1.f - fabsf(2.f * ay - 1.f);
            float dec[kNmOut];
            nm_mlp_wave(static_cast<const NmWeights*>(E.weights), f, dec);
            float tgt[kNmOut];
            if constexpr (kTexel) {
                tgt[0] = la[pa & 0xffu];
                tgt[1] = la[(pa >> 8) & 0xffu];
                tgt[2] = la[(pa >> 16) & 0xffu];
                tgt[3] = ln[pn & 0xffu];
                tgt[4] = ln[pn >> 8];
                tgt[5] = lm[pm & 0xffu];
                tgt[6] = lm[pm >> 8];
            } else {
                nm_target(E.texels, E.textures, S, u, v, lut[1], tgt);
            }
            float e = 0.f;
#pragma unroll
            for (int c = 0; c < kNmOut; ++c) e += (dec[c] - tgt[c]) * (dec[c] - tgt[c]);
            if (x < ta.width && y0 + j < ta.height) err += e;
        }
        const float s = block_sum(err, red_s);
        if (threadIdx.x == 0) E.partial[E.block_base[slot] + blockIdx.x] = s;
        __syncthreads();  // red_s is written again for the next slot
    }
}

// One block per slot: its tiles' sums in FP64, in a fixed order (the host reads one value a slot
// instead of one a tile).
__global__ __launch_bounds__(256) void k_nm_eval_sum(NmEvalLaunch E) {
    __shared__ double red[256];
    for (uint32_t slot = blockIdx.x; slot < E.n_slots; slot += gridDim.x) {
        double s = 0.0;
        for (uint32_t b = E.block_base[slot] + threadIdx.x; b < E.block_base[slot + 1]; b += 256) s += double(E.partial[b]);
        red[threadIdx.x] = s;
        for (uint32_t o = 128; o > 0; o >>= 1) {
            __syncthreads();
            if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        }
        if (threadIdx.x == 0) E.sum[slot] = red[0];
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) void k_nm_points(NmPointLaunch P) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    const uint32_t ii = i < P.n ? i : P.n - 1;  // lanes past the end decode the last point (not stored)
    const uint32_t slot = P.slot[ii];
    const float u = P.uv[2 * size_t(ii)], v = P.uv[2 * size_t(ii) + 1];
    float o[kNmOut];
    if (P.targets) {
        nm_target(P.texels, P.textures, static_cast<const NmSlot*>(P.slots)[slot], u, v, P.srgb_lut, o);
    } else {
        float f[kNmFeat];
        nm_features(P.lat16 + size_t(slot) * P.L * P.L, P.L, u, v, f);
        nm_mlp_wave(static_cast<const NmWeights*>(P.weights), f, o);
    }
    if (i < P.n)
        for (int c = 0; c < kNmOut; ++c) P.out[kNmOut * size_t(i) + c] = o[c];
}

// MFMA-operand form of the MLP (see NmWeights): one wave, lane l writes its own operand entries.
// FP16: every weight rounded to FP16, scales 1.  FP8: each layer's weights (layer 1 with b1 folded
// in) divided by max|w| / 448 and rounded to OCP E4M3 (round to nearest even, the hardware
// conversion), stored as codes; inference widens them to FP16 exactly and the scale multiplies the
// layer's accumulator.
__device__ inline float layer_weight(const float* p, int layer, uint32_t i, uint32_t k) {
    if (layer == 0) return k < uint32_t(kNmIn) ? p[kNmW1 + i * kNmIn + k] : (k == uint32_t(kNmIn) ? p[kNmB1 + i] : 0.f);
    return i < uint32_t(kNmOut) ? p[kNmW2 + i * kNmHidden + k] : 0.f;
}

__device__ void export_weights(const float* p, NmWeights* W, uint32_t fp8) {
    const uint32_t l = threadIdx.x, i = l % 32, hb = l / 32;
    float scale[2] = {1.f, 1.f};
    if (fp8) {
        for (int layer = 0; layer < 2; ++layer) {
            float m = 0.f;
            for (uint32_t e = l; e < 32u * 32u; e += 64) m = fmaxf(m, fabsf(layer_weight(p, layer, e / 32, e % 32)));
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
            scale[layer] = m > 0.f ? m / 448.f : 1.f;
        }
    }
    // the 8 K-values of this lane's entry: layer-1 columns 8 hb + j; layer-2 hidden units nm_hidden(s, hb, j)
    auto put = [&](int layer, uint32_t s, h8& w, uint2& q) {
        uint32_t code[2] = {0u, 0u};
        for (uint32_t j = 0; j < 8; ++j) {
            const uint32_t k = layer == 0 ? 8 * hb + j : nm_hidden(s, hb, j);
            const float v = layer_weight(p, layer, i, k);
            if (fp8) {
                const uint32_t c = uint32_t(__builtin_amdgcn_cvt_pk_fp8_f32(v / scale[layer], 0.f, 0, false)) & 0xffu;
                code[j / 4] |= c << (8 * (j % 4));
                w[j] = _Float16(0.f);
            } else {
                w[j] = _Float16(v);
            }
        }
        q = make_uint2(code[0], code[1]);
    };
    put(0, 0, W->w1[l], W->q1[l]);
    put(1, 0, W->w2[0][l], W->q2[0][l]);
    put(1, 1, W->w2[1][l], W->q2[1][l]);
    if (l < 8) W->b2[l] = l < uint32_t(kNmOut) ? p[kNmB2 + l] : 0.f;
    // FP8: the widened codes carry a factor 2^-8 (nm_widen_e4m3)
    if (l < 2) W->scale[l] = fp8 ? scale[l] * 256.f : 1.f;
    if (l == 0) {
        W->fp8 = fp8 ? 1u : 0u;
        W->first = fp8 ? nm_first_scale(scale[0] * 256.f) : 0x3c003c00u;  // 1 and 1
    }
}

// The inference MLP back in the parameter layout (FP32 values: operand value times layer scale).
__global__ __launch_bounds__(64) void k_nm_unpack_weights(const NmWeights* W, float* p) {
    const uint32_t l = threadIdx.x, i = l % 32, hb = l / 32;
    const bool fp8 = W->fp8 != 0;
    const h8 a1 = fp8 ? nm_widen_e4m3(W->q1[l]) : W->w1[l];
    const h8 a2[2] = {fp8 ? nm_widen_e4m3(W->q2[0][l]) : W->w2[0][l], fp8 ? nm_widen_e4m3(W->q2[1][l]) : W->w2[1][l]};
    for (uint32_t j = 0; j < 8; ++j) {
        const uint32_t k = 8 * hb + j;
        const float v = float(a1[j]) * W->scale[0];
        if (k < uint32_t(kNmIn)) p[kNmW1 + i * kNmIn + k] = v;
        else if (k == uint32_t(kNmIn)) p[kNmB1 + i] = v;
    }
    for (uint32_t s = 0; s < 2; ++s)
        for (uint32_t j = 0; j < 8; ++j)
            if (i < uint32_t(kNmOut)) p[kNmW2 + i * kNmHidden + nm_hidden(s, hb, j)] = float(a2[s][j]) * W->scale[1];
    if (l < uint32_t(kNmOut)) p[kNmB2 + l] = W->b2[l];
}

}  // namespace

hipError_t launch_nm_unpack_weights(const void* weights, float* mlp, hipStream_t s) {
    hipLaunchKernelGGL(k_nm_unpack_weights, dim3(1), dim3(64), 0, s, static_cast<const NmWeights*>(weights), mlp);
    return hipGetLastError();
}

hipError_t launch_nm_init(const NmInitLaunch& l, hipStream_t s) {
    const uint64_t cells = uint64_t(l.n_slots) * l.L * l.L;
    const uint32_t blocks = uint32_t(std::min<uint64_t>((cells + 255) / 256, 65536));
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL(k_nm_init, dim3(blocks), dim3(256), 0, s, l);
    return hipGetLastError();
}

hipError_t launch_nm_gradient(const NmTrainLaunch& l, hipStream_t s) {
    if (l.L > uint32_t(kMaxR)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_nm_step<true>, dim3(l.n_slots), dim3(kStepThreads), 0, s, l);
    hipLaunchKernelGGL(k_nm_mlp<true>, dim3((kNmParamsPad + 63) / 64), dim3(64 * kMlpWaves), 0, s, l);
    return hipGetLastError();
}

hipError_t launch_nm_tables(const NmTrainLaunch& l, hipStream_t s) {
    hipLaunchKernelGGL(k_nm_tables, dim3((kNmParams + 255) / 256), dim3(256), 0, s, l.mlp, l.tables);
    return hipGetLastError();
}

hipError_t launch_nm_steps(NmTrainLaunch l, uint32_t steps, hipStream_t s) {
    if ((1u << l.log2R) > uint32_t(kMaxR) || l.log2R > l.log2L || l.log2R < 1) return hipErrorInvalidValue;
    for (l.step_ahead = 0; l.step_ahead < steps; ++l.step_ahead) {
        hipLaunchKernelGGL(k_nm_step<false>, dim3(l.n_wg), dim3(kStepThreads), 0, s, l);
        hipLaunchKernelGGL(k_nm_mlp<false>, dim3((kNmParamsPad + 63) / 64), dim3(64 * kMlpWaves), 0, s, l);
    }
    hipLaunchKernelGGL(k_nm_advance, dim3(1), dim3(64), 0, s, l.step, steps);
    return hipGetLastError();
}

hipError_t launch_nm_export(const float* lat, uint4* lat16, uint64_t cells, const float* mlp, void* weights,
                            uint32_t fp8, hipStream_t s) {
    const uint32_t blocks = uint32_t(std::min<uint64_t>((cells + 255) / 256, 65536));
    hipLaunchKernelGGL(k_nm_export, dim3(blocks + 1), dim3(256), 0, s, lat, lat16, cells, mlp,
                       static_cast<NmWeights*>(weights), fp8);
    return hipGetLastError();
}

hipError_t launch_nm_eval(const NmEvalLaunch& l, uint32_t max_tiles, bool any_same, bool any_other, hipStream_t s) {
    if (l.n_slots == 0 || max_tiles == 0) return hipSuccess;
    const dim3 grid(max_tiles, min(l.n_slots, 65535u));
    if (any_same) hipLaunchKernelGGL(k_nm_eval<true>, grid, dim3(256), 0, s, l);
    if (any_other) hipLaunchKernelGGL(k_nm_eval<false>, grid, dim3(256), 0, s, l);
    hipLaunchKernelGGL(k_nm_eval_sum, dim3(min(l.n_slots, 65535u)), dim3(256), 0, s, l);
    return hipGetLastError();
}

hipError_t launch_nm_points(const NmPointLaunch& l, hipStream_t s) {
    if (l.n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_nm_points, dim3((l.n + 255) / 256), dim3(256), 0, s, l);
    return hipGetLastError();
}

}  // namespace rsy
