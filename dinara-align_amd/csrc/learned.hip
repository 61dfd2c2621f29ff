// The learned band proposal on MI355X (gfx950): k-mer features of a batch, and a small network that predicts each
// pair's cost from them, trained and run on the device by hand-written bf16 MFMA kernels with fp32 accumulation.
// No counterpart in the reference; the band it proposes is only a first guess: the band certificate still proves
// every result, and a pair it does not prove goes on to the band its cost proves, so every result stays exact.
//
// The network: 288 inputs (258 features and zero padding) -> 256 -> 256 -> 1, ReLU, bf16 weights and activations,
// fp32 accumulation and fp32 master weights updated by Adam. It predicts log(1 + cost).
//
// Products: v_mfma_f32_32x32x8_bf16 over K in steps of 8. Operands as the instruction reads them: lane l holds
// A[l % 32][4(l / 32) .. 4(l / 32) + 3] and B[4(l / 32) .. + 3][l % 32]; the 16 results of lane l are C[8(r / 4) +
// 4(l / 32) + r % 4][l % 32], r = 0..15. So an operand is kept as quads: four consecutive K of one row (or column) in
// 8 bytes, the quads of one K side by side, and a lane reads its operand with one 8-byte load, 32 lanes 256 bytes in a
// row; and a lane's results are quads of four consecutive rows, which is how the products over rows (the weights'
// gradients) read them. A training step is two launches: one takes 32 rows a workgroup through both layers, the output
// and back to the first layer's gradients (everything that stays within a row), the other makes every sum over rows and
// updates the weights with it. Every sum is taken in one fixed order (products by K, the others row by row), so a
// network's numbers do not depend on how the work is split.

#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <type_traits>
#include <vector>

#include "../../include/dinara.h"
#include "device.h"
#include "learned.h"

namespace dinara {

// ------------------------------------------------------------------ features

// 4-mer counts of 64 slots a workgroup, a thread a slot, in LDS (the thread's own 257-word row: the padding word
// spreads the rows over the banks). A 2-bit tape is read a word (16 letters) at a time: the 16 windows that end in
// the word come from the word and the one before it as 64 bits, and each is counted with an LDS add whose result
// is not waited for. The windows are counted by their tape bits (first letter lowest); a forward 4-mer code puts
// the first letter highest, so a forward tape's counts are read back with the four 2-bit fields reversed. The
// feature rows are then written a slot at a time by the whole wave, 64 consecutive floats a store.
__global__ __launch_bounds__(64) void kmer_features(Tape tape, int slots, int reversed, float *out) {
    constexpr int ROW = 257;
    __shared__ int32_t hist[64 * ROW];
    const int t = threadIdx.x, slot = blockIdx.x * 64 + t;
    int32_t *mine = hist + t * ROW;
    for (int k = 0; k < 256; ++k) mine[k] = 0;
    if (slot < slots) {
        const int g = slot >> 6, col = slot & 63;
        const uint32_t *ref_words = tape.words + tape.group_base[g] + col;
        const uint32_t *qry_words = ref_words + (size_t)tape.group_ref_words[g] * 64;
        const int bits = tape.bits, per = 32 / bits;
        auto count = [&](const uint32_t *words, int len, int delta) {
            if (bits == 2) {
                // Eight words a step, the next eight loaded while these are counted.
                const int total = (len + 15) >> 4;
                auto load = [&](uint32_t (&to)[8], int w0) {
#pragma unroll
                    for (int k = 0; k < 8; ++k) to[k] = w0 + k < total ? words[(size_t)(w0 + k) * 64] : 0u;
                };
                uint32_t now[8], next[8];
                load(now, 0);
                uint32_t before = 0;
                for (int w0 = 0; w0 < total; w0 += 8) {
                    load(next, w0 + 8);
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        const int w = w0 + k;
                        const uint64_t pair = (uint64_t)before | ((uint64_t)now[k] << 32);
                        // Window j starts at letter 16w + j - 3 and ends at letter 16w + j.
                        const int first = w == 0 ? 3 : 0, last = len - 16 * w;
#pragma unroll
                        for (int j = 0; j < 16; ++j) {
                            if (j >= first && j < last) atomicAdd(&mine[(uint32_t)((pair >> (26 + 2 * j)) & 255u)], delta);
                        }
                        before = now[k];
                    }
#pragma unroll
                    for (int k = 0; k < 8; ++k) now[k] = next[k];
                }
                return;
            }
            uint32_t window = 0;  // the last four letters, first lowest
            int seen = 0;
            for (int w = 0; w * per < len; ++w) {
                uint32_t word = words[(size_t)w * 64];
                const int here = min(per, len - w * per);
                for (int i = 0; i < here; ++i) {
                    window = (window >> 2) | ((word & 3u) << 6);
                    word >>= bits;
                    if (++seen >= 4) atomicAdd(&mine[window], delta);
                }
            }
        };
        count(ref_words, tape.rows[slot], 1);
        count(qry_words, tape.cols[slot], -1);
    }
    __syncthreads();
    // A reversed tape holds each sequence back to front: its windows' tape bits are then the forward codes.
    const int first = blockIdx.x * 64, here = min(64, slots - first);
    for (int s = 0; s < here; ++s) {
        const int n = tape.rows[first + s], m = tape.cols[first + s];
        const float scale = 8.0f / sqrtf(1.0f + (float)n + (float)m);
        float *row = out + (size_t)(first + s) * FEATURE_STRIDE;
        for (int k = t; k < FEATURE_STRIDE; k += 64) {
            float v = 0.0f;
            if (k < 256) {
                const int at = reversed ? k : ((k & 3) << 6) | ((k & 12) << 2) | ((k & 48) >> 2) | (k >> 6);
                v = (float)hist[s * ROW + at] * scale;
            } else if (k == 256) {
                v = (logf(1.0f + (float)n) - 7.0f) * 0.5f;
            } else if (k == 257) {
                v = (logf(1.0f + (float)m) - 7.0f) * 0.5f;
            }
            row[k] = v;
        }
    }
}

void launch_features(const Tape &tape, int slots, int reversed, float *out, hipStream_t stream) {
    if (slots <= 0) return;
    hipLaunchKernelGGL(kmer_features, dim3((slots + 63) / 64), dim3(64), 0, stream, tape, slots, reversed, out);
}

// ------------------------------------------------------------------ bf16 and the MFMA product

// fp32 to bf16, round to nearest even (finite values; the network never makes others).
__device__ inline uint16_t to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ inline float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int HIDDEN = 256;
constexpr int IN_QUADS = FEATURE_STRIDE / 4, HIDDEN_QUADS = HIDDEN / 4;
// The flat weights (as the C ABI gives them) and their bf16 copies: w1 and w2 as quads along their rows (the forward
// products' K), w2 again as quads along its columns (the backward product's K), w3 as it is.
constexpr int W1 = 0, B1 = W1 + FEATURE_STRIDE * HIDDEN, W2 = B1 + HIDDEN, B2 = W2 + HIDDEN * HIDDEN,
              W3 = B2 + HIDDEN, B3 = W3 + HIDDEN, WEIGHTS = B3 + 1;
constexpr int W1_QUADS = 0, W2_QUADS = W1_QUADS + FEATURE_STRIDE * HIDDEN, W2T_QUADS = W2_QUADS + HIDDEN * HIDDEN,
              W3_COPY = W2T_QUADS + HIDDEN * HIDDEN, COPIES = W3_COPY + HIDDEN;

// Where w[k][j] of a `HIDDEN`-column matrix is among its quads along k.
__host__ __device__ constexpr int quad_place(int k, int j) { return ((k >> 2) * HIDDEN + j) * 4 + (k & 3); }

// What a training step reads and leaves. `x` (rows x FEATURE_STRIDE fp32) and `targets` are read at `index` (null: in
// order); the first `count` of the step's rows are real. For the sums over rows: x, both layers' activations and their
// gradients as bf16 quads of four rows, and per row the output's gradient and squared error.
struct StepArgs {
    const float *x, *targets;
    const int32_t *index;
    int count, rows;
    const float *weights;
    const uint16_t *copies;
    bf16x4 *x_quads, *a1_quads, *a2_quads, *dz1_quads, *dz2_quads;
    float *dy, *sq, *y;
};

// Quads of a 32-row block in LDS, K quad q of row i at [q][i]: a row of 33, so that the lanes that write a column's
// quads fall in different banks.
constexpr int LDS_ROW = 33;

// One wave's 32 x 32 tile of A (32 rows, quads in LDS) . B (columns `column`, quads of HIDDEN columns in global
// memory), K = 8 STEPS: B's operands are loaded GROUP steps at once.
template <int STEPS, int GROUP>
__device__ __forceinline__ f32x16 block_product(const bf16x4 *a, const bf16x4 *b, int column, int lane) {
    static_assert(STEPS % GROUP == 0, "whole groups");
    const int half = lane >> 5, row = lane & 31;
    f32x16 acc = {};
    for (int s0 = 0; s0 < STEPS; s0 += GROUP) {
        bf16x4 vb[GROUP];
#pragma unroll
        for (int u = 0; u < GROUP; ++u) vb[u] = b[(size_t)(2 * (s0 + u) + half) * HIDDEN + column];
#pragma unroll
        for (int u = 0; u < GROUP; ++u)
            acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a[(2 * (s0 + u) + half) * LDS_ROW + row], vb[u], acc, 0, 0, 0);
    }
    return acc;
}

// A lane's value of row i, column j as an element of the next product's A quads.
__device__ __forceinline__ void put_quad(bf16x4 *quads, int i, int j, uint16_t v) {
    reinterpret_cast<uint16_t *>(quads)[((j >> 2) * LDS_ROW + i) * 4 + (j & 3)] = v;
}

// 32 rows a workgroup, a wave a 32-column tile: the forward pass and the output, and (TRAIN) the loss's gradient back
// to the first layer. Bounded by its chains (36 and 32 matrix steps of 64 cycles, the output's 256 additions a row):
// 4,096 rows took 15 us a product and 150 for the output as kernels of their own, each activation out to memory and
// back; here the activations pass through LDS, 25 us for all of it.
template <bool TRAIN>
__global__ __launch_bounds__(512) void network_rows(StepArgs a) {
    __shared__ bf16x4 in_quads[IN_QUADS * LDS_ROW], act[HIDDEN_QUADS * LDS_ROW];
    __shared__ float slope[32];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int i0 = blockIdx.x * 32, j = wave * 32 + (lane & 31), half = lane >> 5;
    for (int at = t; at < 32 * IN_QUADS; at += 512) {
        const int i = at / IN_QUADS, q = at % IN_QUADS, r = i0 + i;
        float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
        if (r < a.count)
            f = *reinterpret_cast<const float4 *>(a.x + (size_t)(a.index ? a.index[r] : r) * FEATURE_STRIDE + 4 * q);
        in_quads[q * LDS_ROW + i] =
            bf16x4{(short)to_bf16(f.x), (short)to_bf16(f.y), (short)to_bf16(f.z), (short)to_bf16(f.w)};
    }
    __syncthreads();
    if (TRAIN) {
        const short *x = reinterpret_cast<const short *>(in_quads);
        for (int at = t; at < 8 * FEATURE_STRIDE; at += 512) {
            const int i = 4 * (at / FEATURE_STRIDE), k = at % FEATURE_STRIDE;
            const short *from = x + ((k >> 2) * LDS_ROW + i) * 4 + (k & 3);
            a.x_quads[(size_t)((i0 + i) >> 2) * FEATURE_STRIDE + k] = bf16x4{from[0], from[4], from[8], from[12]};
        }
    }
    const bf16x4 *const copies = reinterpret_cast<const bf16x4 *>(a.copies);
    // A layer's bias and ReLU: bf16 activations into `to`, and (TRAIN) four rows at a time into `rows_to`.
    const auto activate = [&](f32x16 &z, const float *bias, bf16x4 *to, bf16x4 *rows_to) __attribute__((always_inline)) {
        const float b = bias[j];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            bf16x4 four;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = z[4 * q + e] + b;
                z[4 * q + e] = v;
                four[e] = (short)to_bf16(v > 0.0f ? v : 0.0f);
                put_quad(to, 8 * q + 4 * half + e, j, (uint16_t)four[e]);
            }
            if (TRAIN) rows_to[(size_t)((i0 + 8 * q + 4 * half) >> 2) * HIDDEN + j] = four;
        }
    };
    f32x16 z1 = block_product<IN_QUADS / 2, 12>(in_quads, copies + W1_QUADS / 4, j, lane);
    activate(z1, a.weights + B1, act, a.a1_quads);
    uint32_t live1 = 0;  // the first layer's units the gradient passes
#pragma unroll
    for (int r = 0; r < 16; ++r) live1 |= (z1[r] <= 0.0f ? 0u : 1u) << r;
    __syncthreads();
    f32x16 z2 = block_product<HIDDEN_QUADS / 2, 16>(act, copies + W2_QUADS / 4, j, lane);
    __syncthreads();
    activate(z2, a.weights + B2, act, a.a2_quads);
    __syncthreads();
    // The output: a lane a row, summed in column order.
    const uint16_t *const w3 = a.copies + W3_COPY;
    if (t < 32) {
        const int r = i0 + t;
        float s = a.weights[B3];
#pragma unroll 16
        for (int q = 0; q < HIDDEN_QUADS; ++q) {
            const bf16x4 four = act[q * LDS_ROW + t];
#pragma unroll
            for (int e = 0; e < 4; ++e) s += from_bf16((uint16_t)four[e]) * from_bf16(w3[4 * q + e]);
        }
        if (!TRAIN) {
            if (r < a.count) a.y[r] = s;
        } else {
            const float target = r < a.count ? a.targets[a.index ? a.index[r] : r] : 0.0f;
            const float d = r < a.count ? 2.0f * (s - target) / (float)a.count : 0.0f;
            a.dy[r] = slope[t] = d;
            a.sq[r] = r < a.count ? (s - target) * (s - target) : 0.0f;
        }
    }
    if constexpr (TRAIN) {
        __syncthreads();
        // dZ2 = dy w3 where Z2 > 0, dZ1 = dZ2 W2^T where Z1 > 0.
        const float w = from_bf16(w3[j]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            bf16x4 four;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int i = 8 * q + 4 * half + e;
                four[e] = (short)to_bf16(z2[4 * q + e] > 0.0f ? slope[i] * w : 0.0f);
                put_quad(act, i, j, (uint16_t)four[e]);
            }
            a.dz2_quads[(size_t)((i0 + 8 * q + 4 * half) >> 2) * HIDDEN + j] = four;
        }
        __syncthreads();
        const f32x16 dz1 = block_product<HIDDEN_QUADS / 2, 16>(act, copies + W2T_QUADS / 4, j, lane);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            bf16x4 four;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                four[e] = (short)to_bf16((live1 >> (4 * q + e)) & 1u ? dz1[4 * q + e] : 0.0f);
            a.dz1_quads[(size_t)((i0 + 8 * q + 4 * half) >> 2) * HIDDEN + j] = four;
        }
    }
}

// One Adam step on a parameter: m, v the moments, `scale` = lr * sqrt(1 - b2^t) / (1 - b1^t).
struct AdamArgs {
    float *w, *m, *v;
    uint16_t *copies;
    float b1, b2, scale, eps;
};
__device__ __forceinline__ float adam(const AdamArgs &p, int at, float gi) {
    const float mi = p.b1 * p.m[at] + (1.0f - p.b1) * gi;
    const float vi = p.b2 * p.v[at] + (1.0f - p.b2) * gi * gi;
    p.m[at] = mi;
    p.v[at] = vi;
    const float wi = p.w[at] - p.scale * mi / (sqrtf(vi) + p.eps);
    p.w[at] = wi;
    return wi;
}

// A chain of `steps` in order, `load(bank, place, step)` AHEAD steps before `use(bank, place)`: two banks of registers
// take turns, the loads of one all made before the other is used (the fence keeps them there: left to itself the
// compiler moved each load behind its bank's last use, and every bank waited for memory). Loads past the end read the
// last step again.
constexpr int AHEAD = 16;
template <typename Load, typename Use>
__device__ __forceinline__ void ahead(int steps, Load load, Use use) {
    const auto fill = [&](auto bank, int from) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) load(bank, u, from + u < steps ? from + u : steps - 1);
        __builtin_amdgcn_sched_barrier(0);
    };
    const auto drain = [&](auto bank, int left) __attribute__((always_inline)) {
        if (left >= AHEAD) {
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) use(bank, u);
        } else {
#pragma unroll
            for (int u = 0; u < AHEAD; ++u)
                if (u < left) use(bank, u);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const std::integral_constant<int, 0> one;
    const std::integral_constant<int, 1> other;
    fill(one, 0);
    for (int step = 0; step < steps; step += 2 * AHEAD) {
        fill(other, step + AHEAD);
        drain(one, steps - step);
        fill(one, step + 2 * AHEAD);
        drain(other, steps - step - AHEAD);
    }
}

// One column's sum over `quads` quads of rows, each row times its weight or as it is, row by row.
template <bool WEIGHTED>
__device__ __forceinline__ float column_sum(const bf16x4 *from, const float *weights, int quads) {
    const float4 *by = reinterpret_cast<const float4 *>(weights);
    float s = 0.0f;
    bf16x4 v[2][AHEAD];
    float4 w[2][AHEAD];
    ahead(quads,
          [&](auto bank, int u, int q) __attribute__((always_inline)) {
              v[bank.value][u] = from[(size_t)q * HIDDEN];
              if (WEIGHTED) w[bank.value][u] = by[q];
          },
          [&](auto bank, int u) __attribute__((always_inline)) {
              const bf16x4 four = v[bank.value][u];
              const float4 f = WEIGHTED ? w[bank.value][u] : make_float4(1.f, 1.f, 1.f, 1.f);
              s += f.x * from_bf16((uint16_t)four[0]);
              s += f.y * from_bf16((uint16_t)four[1]);
              s += f.z * from_bf16((uint16_t)four[2]);
              s += f.w * from_bf16((uint16_t)four[3]);
          });
    return s;
}

// Every sum over a step's rows, a wave each: the 32 x 32 tiles of dW1 = X^T dZ1 and dW2 = A1^T dZ2, 64 columns of db1,
// db2 or dw3 = A2^T dy, and db3 with the loss. UPDATE takes an Adam step with each sum, else it is left in `grad`.
// Each sum is one chain over the rows (a matrix step of 64 cycles every 8, an addition each), so the launch takes what
// its longest chain does: at 4,096 rows the products took 279 us each, a column's sums 633 and a row's 149, loading one
// value at a time where the chain waited for it; with quads loaded AHEAD steps before, 39 us for all of them together.
constexpr int TILES1 = FEATURE_STRIDE / 32 * (HIDDEN / 32), TILES2 = HIDDEN / 32 * (HIDDEN / 32),
              COLUMN_WAVES = HIDDEN / 64;
template <bool UPDATE>
__global__ __launch_bounds__(64) void network_sums(StepArgs a, float *grad, float *loss, AdamArgs p) {
    const int lane = threadIdx.x, quads = a.rows >> 2;
    int at = (int)blockIdx.x;
    if (at < TILES1 + TILES2) {
        const bool first = at < TILES1;
        if (!first) at -= TILES1;
        const int i0 = at / (HIDDEN / 32) * 32, j0 = at % (HIDDEN / 32) * 32, half = lane >> 5, place = lane & 31;
        const int width = first ? FEATURE_STRIDE : HIDDEN;
        const bf16x4 *left = (first ? a.x_quads : a.a1_quads) + (size_t)half * width + i0 + place;
        const bf16x4 *right = (first ? a.dz1_quads : a.dz2_quads) + (size_t)half * HIDDEN + j0 + place;
        f32x16 acc = {};
        const int steps = quads >> 1;  // a multiple of 4
        bf16x4 va[2][AHEAD], vb[2][AHEAD];
        ahead(steps,
              [&](auto bank, int u, int step) __attribute__((always_inline)) {
                  va[bank.value][u] = left[(size_t)step * 2 * width];
                  vb[bank.value][u] = right[(size_t)step * 2 * HIDDEN];
              },
              [&](auto bank, int u) __attribute__((always_inline)) {
                  acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(va[bank.value][u], vb[bank.value][u], acc, 0, 0, 0);
              });
        const int j = j0 + place, base = first ? W1 : W2;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = i0 + 8 * q + 4 * half;
            bf16x4 four;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int place_of = base + (i + e) * HIDDEN + j;
                if (UPDATE) {
                    four[e] = (short)to_bf16(adam(p, place_of, acc[4 * q + e]));
                    if (!first) p.copies[W2T_QUADS + quad_place(j, i + e)] = (uint16_t)four[e];
                } else {
                    grad[place_of] = acc[4 * q + e];
                }
            }
            if (UPDATE)
                *reinterpret_cast<bf16x4 *>(p.copies + (first ? W1_QUADS : W2_QUADS) + quad_place(i, j)) = four;
        }
        return;
    }
    at -= TILES1 + TILES2;
    if (at < 3 * COLUMN_WAVES) {
        // 64 columns of db1, db2 or dw3, the last with each row's dy.
        const int which = at / COLUMN_WAVES, j = at % COLUMN_WAVES * 64 + lane;
        const bf16x4 *from = (which == 0 ? a.dz1_quads : which == 1 ? a.dz2_quads : a.a2_quads) + j;
        const float s = which == 2 ? column_sum<true>(from, a.dy, quads) : column_sum<false>(from, a.dy, quads);
        const int place_of = (which == 0 ? B1 : which == 1 ? B2 : W3) + j;
        if (UPDATE) {
            const float wi = adam(p, place_of, s);
            if (which == 2) p.copies[W3_COPY + j] = to_bf16(wi);
        } else {
            grad[place_of] = s;
        }
        return;
    }
    // The output's gradient (lane 0) and the squared errors (lane 1), row by row.
    if (lane > 1) return;
    const float4 *from = reinterpret_cast<const float4 *>(lane == 0 ? a.dy : a.sq);
    float s = 0.0f;
    float4 v[2][AHEAD];
    ahead(quads, [&](auto bank, int u, int q) __attribute__((always_inline)) { v[bank.value][u] = from[q]; },
          [&](auto bank, int u) __attribute__((always_inline)) {
              s += v[bank.value][u].x;
              s += v[bank.value][u].y;
              s += v[bank.value][u].z;
              s += v[bank.value][u].w;
          });
    if (lane == 1)
        *loss = s;
    else if (UPDATE)
        adam(p, B3, s);
    else
        grad[B3] = s;
}

// The bf16 copies of the fp32 weights.
__global__ void copy_weights(const float *w, uint16_t *copies) {
    const int at = blockIdx.x * 256 + threadIdx.x;
    if (at < B1) {
        copies[W1_QUADS + quad_place(at / HIDDEN, at % HIDDEN)] = to_bf16(w[W1 + at]);
    } else if (at >= W2 && at < B2) {
        const int i = (at - W2) / HIDDEN, j = (at - W2) % HIDDEN;
        copies[W2_QUADS + quad_place(i, j)] = copies[W2T_QUADS + quad_place(j, i)] = to_bf16(w[at]);
    } else if (at >= W3 && at < B3) {
        copies[W3_COPY + at - W3] = to_bf16(w[at]);
    }
}

}  // namespace dinara

using namespace dinara;

// ------------------------------------------------------------------ the network and its C ABI

struct dinara_mlp {
    DeviceContext *ctx = nullptr;
    int rows_cap = 0;   // rows the work buffers hold
    int64_t step = 0;   // Adam's step count
    // fp32 master weights, gradients and Adam moments (flat: w1, b1, w2, b2, w3, b3), and the weights' bf16 copies
    DeviceBuffer master, copies, grad, m1, m2;
    // per-step work
    DeviceBuffer x_quads, a1_quads, a2_quads, dz1_quads, dz2_quads, dy, sq;
    DeviceBuffer features, targets, index, loss;
    DeviceBuffer predicted;   // the prediction's output for `dinara_mlp_predict`
};

namespace {

using Net = dinara_mlp;

float *f32(DeviceBuffer &b, size_t offset = 0) { return static_cast<float *>(b.ptr) + offset; }

bool reserve_rows(Net *net, int rows) {
    if (rows <= net->rows_cap) return true;
    const size_t r = (size_t)rows;
    for (DeviceBuffer *b : {&net->a1_quads, &net->a2_quads, &net->dz1_quads, &net->dz2_quads})
        if (!b->reserve(r * HIDDEN * 2)) return false;
    if (!net->x_quads.reserve(r * FEATURE_STRIDE * 2) || !net->dy.reserve(r * 4) || !net->sq.reserve(r * 4)) return false;
    net->rows_cap = rows;
    return true;
}

StepArgs step_args(Net *net, const float *x, int count, int rows) {
    StepArgs a{};
    a.x = x;
    a.count = count;
    a.rows = rows;
    a.weights = f32(net->master);
    a.copies = static_cast<const uint16_t *>(net->copies.ptr);
    const auto quads = [](DeviceBuffer &b) { return static_cast<bf16x4 *>(b.ptr); };
    a.x_quads = quads(net->x_quads);
    a.a1_quads = quads(net->a1_quads);
    a.a2_quads = quads(net->a2_quads);
    a.dz1_quads = quads(net->dz1_quads);
    a.dz2_quads = quads(net->dz2_quads);
    a.dy = f32(net->dy);
    a.sq = f32(net->sq);
    return a;
}

// A step's two launches over `a.rows` rows (a multiple of 32); its summed squared error into *loss.
template <bool UPDATE>
void launch_step(Net *net, const StepArgs &a, float *loss, const AdamArgs &p) {
    hipStream_t s = net->ctx->stream;
    hipLaunchKernelGGL((network_rows<true>), dim3(a.rows / 32), dim3(512), 0, s, a);
    hipLaunchKernelGGL((network_sums<UPDATE>), dim3(TILES1 + TILES2 + 3 * COLUMN_WAVES + 1), dim3(64), 0, s, a,
                       f32(net->grad), loss, p);
}

void refresh_copies(Net *net) {
    hipLaunchKernelGGL(copy_weights, dim3((WEIGHTS + 255) / 256), dim3(256), 0, net->ctx->stream, f32(net->master),
                       static_cast<uint16_t *>(net->copies.ptr));
}

}  // namespace

int64_t mlp_predict_into(dinara_mlp *net, const float *features, int64_t rows, float *out) {
    if (!net) return DINARA_INVALID_MODE;
    DeviceGuard guard(net->ctx);
    constexpr int64_t most = int64_t(1) << 22;  // rows a launch: row numbers times the stride stay in 32 bits
    for (int64_t first = 0; first < rows; first += most) {
        const int count = (int)std::min(most, rows - first);
        StepArgs a = step_args(net, features + first * FEATURE_STRIDE, count, count);
        a.y = out + first;
        hipLaunchKernelGGL((network_rows<false>), dim3((count + 31) / 32), dim3(512), 0, net->ctx->stream, a);
    }
    return hipPeekAtLastError() == hipSuccess ? 0 : DINARA_OUT_OF_MEMORY;
}

int64_t mlp_predict_device(dinara_mlp *net, const float *features, int64_t rows, float *out) {
    if (!net) return DINARA_INVALID_MODE;
    if (rows <= 0) return 0;
    DeviceGuard guard(net->ctx);
    if (!net->predicted.reserve((size_t)rows * 4)) return DINARA_OUT_OF_MEMORY;
    if (const int64_t code = mlp_predict_into(net, features, rows, f32(net->predicted))) return code;
    return net->predicted.read(net->ctx, out, (size_t)rows * 4) ? 0 : DINARA_OUT_OF_MEMORY;
}

extern "C" {

dinara_mlp *dinara_mlp_new(int64_t gpu, uint64_t seed) {
    DeviceContext *ctx = device_context(gpu);
    if (!ctx) return nullptr;
    DeviceGuard guard(ctx);
    auto *net = new Net();
    net->ctx = ctx;
    // He-normal weights for the ReLU layers (the padding inputs' rows zero), a small output layer, zero biases.
    std::vector<float> w(WEIGHTS, 0.0f);
    std::mt19937_64 rng(seed);
    std::normal_distribution<float> n1(0.0f, std::sqrt(2.0f / FEATURES)), n2(0.0f, std::sqrt(2.0f / (float)HIDDEN)),
        n3(0.0f, std::sqrt(1.0f / (float)HIDDEN));
    for (size_t k = 0; k < (size_t)FEATURES * HIDDEN; ++k) w[W1 + k] = n1(rng);
    for (size_t k = 0; k < (size_t)HIDDEN * HIDDEN; ++k) w[W2 + k] = n2(rng);
    for (size_t k = 0; k < (size_t)HIDDEN; ++k) w[W3 + k] = n3(rng);
    w[B3] = 7.0f;  // log(1 + cost) of a typical pair, where training starts
    const size_t bytes = (size_t)WEIGHTS * 4;
    std::vector<float> zero(WEIGHTS, 0.0f);
    if (!net->master.upload(ctx, w.data(), bytes) || !net->copies.reserve((size_t)COPIES * 2) ||
        !net->grad.reserve(bytes) || !net->m1.upload(ctx, zero.data(), bytes) ||
        !net->m2.upload(ctx, zero.data(), bytes)) {
        delete net;
        return nullptr;
    }
    refresh_copies(net);
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) {
        delete net;
        return nullptr;
    }
    return net;
}

void dinara_mlp_free(dinara_mlp *net) {
    if (!net) return;
    DeviceGuard guard(net->ctx);
    delete net;
}

int64_t dinara_mlp_parameter_count(dinara_mlp *net) { return net ? (int64_t)WEIGHTS : 0; }

// The fp32 master weights, flat: w1 (288 x 256, row k input k), b1 (256), w2 (256 x 256), b2, w3 (256), b3 (1).
int64_t dinara_mlp_get_weights(dinara_mlp *net, float *out) {
    if (!net) return DINARA_INVALID_MODE;
    DeviceGuard guard(net->ctx);
    return net->master.read(net->ctx, out, (size_t)WEIGHTS * 4) ? 0 : DINARA_OUT_OF_MEMORY;
}

int64_t dinara_mlp_set_weights(dinara_mlp *net, const float *in) {
    if (!net) return DINARA_INVALID_MODE;
    DeviceGuard guard(net->ctx);
    if (!net->master.write(net->ctx, in, (size_t)WEIGHTS * 4)) return DINARA_OUT_OF_MEMORY;
    refresh_copies(net);
    return hipStreamSynchronize(net->ctx->stream) == hipSuccess ? 0 : DINARA_OUT_OF_MEMORY;
}

// The gradients of the mean squared error over `rows` rows (features FEATURE_STRIDE floats a row, targets one a
// row) at the current weights, flat as the weights, and the loss.
int64_t dinara_mlp_gradients(dinara_mlp *net, int64_t rows, const float *features, const float *targets,
                             float *gradients, double *loss) {
    if (!net || rows <= 0) return DINARA_INVALID_MODE;
    DeviceGuard guard(net->ctx);
    const int64_t padded = (rows + 31) / 32 * 32;
    if (padded > INT32_MAX || !reserve_rows(net, (int)padded) || !net->loss.reserve(4) ||
        !net->features.upload(net->ctx, features, (size_t)rows * FEATURE_STRIDE * 4) ||
        !net->targets.upload(net->ctx, targets, (size_t)rows * 4))
        return DINARA_OUT_OF_MEMORY;
    StepArgs a = step_args(net, f32(net->features), (int)rows, (int)padded);
    a.targets = f32(net->targets);
    launch_step<false>(net, a, f32(net->loss), AdamArgs{});
    float sq = 0;
    if (hipPeekAtLastError() != hipSuccess || !net->grad.read(net->ctx, gradients, (size_t)WEIGHTS * 4) ||
        !net->loss.read(net->ctx, &sq, 4))
        return DINARA_OUT_OF_MEMORY;
    if (loss) *loss = sq / (double)rows;
    return 0;
}

// Predictions (log(1 + cost)) for `rows` rows.
int64_t dinara_mlp_predict(dinara_mlp *net, int64_t rows, const float *features, float *out) {
    if (!net) return DINARA_INVALID_MODE;
    if (rows <= 0) return 0;
    DeviceGuard guard(net->ctx);
    constexpr int64_t most = int64_t(1) << 20;  // rows on the device at once (1.2 GB of features)
    for (int64_t first = 0; first < rows; first += most) {
        const int64_t count = std::min(most, rows - first);
        if (!net->features.upload(net->ctx, features + first * FEATURE_STRIDE, (size_t)count * FEATURE_STRIDE * 4))
            return DINARA_OUT_OF_MEMORY;
        if (const int64_t code = mlp_predict_device(net, f32(net->features), count, out + first)) return code;
    }
    return 0;
}

// Trains on `rows` rows for `epochs` passes in shuffled batches of `batch` rows (a multiple of 32) by Adam at
// learning rate `lr`: every step's forward, backward and update on the device, the host waiting once an epoch (for the
// steps' losses). Writes the last epoch's mean loss.
int64_t dinara_mlp_train(dinara_mlp *net, int64_t rows, const float *features, const float *targets, int64_t epochs,
                         int64_t batch, double lr, uint64_t seed, double *final_loss) {
    if (!net || rows <= 0 || batch <= 0 || batch % 32 != 0) return DINARA_INVALID_MODE;
    DeviceContext *ctx = net->ctx;
    DeviceGuard guard(ctx);
    const int64_t steps = (rows + batch - 1) / batch;
    if (batch > INT32_MAX || !reserve_rows(net, (int)batch) || !net->loss.reserve((size_t)steps * 4) ||
        !net->features.upload(ctx, features, (size_t)rows * FEATURE_STRIDE * 4) ||
        !net->targets.upload(ctx, targets, (size_t)rows * 4) || !net->index.reserve((size_t)rows * 4))
        return DINARA_OUT_OF_MEMORY;
    std::vector<int32_t> order((size_t)rows);
    for (int64_t i = 0; i < rows; ++i) order[i] = (int32_t)i;
    std::mt19937_64 rng(seed);
    std::vector<float> losses((size_t)steps);
    double epoch_loss = 0;
    AdamArgs p{};
    p.w = f32(net->master);
    p.m = f32(net->m1);
    p.v = f32(net->m2);
    p.copies = static_cast<uint16_t *>(net->copies.ptr);
    p.b1 = 0.9f;
    p.b2 = 0.999f;
    p.eps = 1e-8f;
    for (int64_t e = 0; e < epochs; ++e) {
        std::shuffle(order.begin(), order.end(), rng);
        if (!net->index.write(ctx, order.data(), order.size() * 4)) return DINARA_OUT_OF_MEMORY;
        for (int64_t at = 0; at < steps; ++at) {
            const int64_t first = at * batch;
            StepArgs a = step_args(net, f32(net->features), (int)std::min<int64_t>(batch, rows - first), (int)batch);
            a.targets = f32(net->targets);
            a.index = static_cast<const int32_t *>(net->index.ptr) + first;
            ++net->step;
            const double bias1 = 1.0 - std::pow((double)p.b1, (double)net->step);
            const double bias2 = 1.0 - std::pow((double)p.b2, (double)net->step);
            p.scale = (float)(lr * std::sqrt(bias2) / bias1);
            launch_step<true>(net, a, f32(net->loss) + at, p);
        }
        if (hipPeekAtLastError() != hipSuccess || !net->loss.read(ctx, losses.data(), losses.size() * 4))
            return DINARA_OUT_OF_MEMORY;
        double sum = 0;
        for (float sq : losses) sum += sq;
        epoch_loss = sum / (double)rows;
    }
    if (final_loss) *final_loss = epoch_loss;
    return 0;
}

}  // extern "C"
