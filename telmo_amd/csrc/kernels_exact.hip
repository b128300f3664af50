// The exact kernel: the reference's fused arithmetic on the GPU, for validation and for callers
// that need bit-identity with telmo's SIMD CPU kernels, and the products no integer path takes
// (f32, f16 and bf16 weights, row-major f32 right-hand sides).
//
// Every output is acc = fmaf(a[r][i], widen(w)[o][i], acc) for i = 0..k-1 in order
// (src/kernels/avx512.rs:70-105 and 156-213: input-order fused sums), with widen as
// src/kernels/scalar.rs:54-107 (int8: one rounded product q * scale), then the shared epilogue,
// which uses the reference's SIMD exp. Any precision; weights in the device layout.
#include "tg_internal.hpp"

namespace tg {

typedef float v4f __attribute__((ext_vector_type(4)));

namespace {

__device__ __forceinline__ float half_to_float(uint16_t h) {
    const uint32_t sign = (uint32_t)(h & 0x8000) << 16;
    const uint32_t exp = (h >> 10) & 0x1f, man = h & 0x3ff;
    if (exp == 0) {
        if (man == 0) return __uint_as_float(sign);
        const float v = (float)man * (1.0f / 16777216.0f);
        return sign ? -v : v;
    }
    if (exp == 0x1f) return __uint_as_float(sign | 0x7f800000u | (man ? 0x400000u | (man << 13) : 0u));
    return __uint_as_float(sign | ((exp + 112) << 23) | (man << 13));
}

__device__ __forceinline__ float widen_one(const uint8_t *__restrict__ wv, const float *__restrict__ scales,
                                           uint32_t prec, size_t k, size_t ps, size_t bs, size_t p, int j, size_t i) {
    switch (prec) {
    case F32: return reinterpret_cast<const float *>(wv)[(p * k + i) * PANEL + j];
    case F16: return half_to_float(reinterpret_cast<const uint16_t *>(wv)[(p * k + i) * PANEL + j]);
    case BF16: return __uint_as_float((uint32_t)reinterpret_cast<const uint16_t *>(wv)[(p * k + i) * PANEL + j] << 16);
    default: {
        const size_t t = i / KBLK, g = (i % KBLK) / 16, ii = i % 16;
        const int8_t q = (int8_t)wv[p * ps + t * bs + (g * 16 + j) * 16 + ii];
        const float s = prec == INT8 ? scales[p * PANEL + j]
                                     : scales[(p * div_ceil(k, Q8_BLOCK) + i / Q8_BLOCK) * PANEL + j];
        return (float)q * s;
    }
    }
}

// The accuracy guard's fix-up (RowGuard): the exact kernel's sums (one lane per output, since flagged
// rows are few) and epilogue for the flagged rows of a product the fast path has just written, over
// every output column. Workgroup (x, y) takes the 64 columns 64 x .. and the rows of chunk y; its
// wavefronts read the chunk's flags 64 at a time and take the flagged rows in turn (wavefront w the
// w-th, w + 4-th, ... of each group of 64). A flagged row's old outputs come from save (kept by the
// quantiser) when the epilogue accumulates.
__global__ __launch_bounds__(256) void exact_rows_kernel(const float *__restrict__ a, size_t lda, int m, int k,
                                                         const uint8_t *__restrict__ wv,
                                                         const float *__restrict__ scales, uint32_t prec, int N,
                                                         size_t ps, size_t bs, float *__restrict__ c, size_t ldc,
                                                         const float *__restrict__ bias, uint32_t act, float escale,
                                                         int accumulate, const int32_t *__restrict__ flags,
                                                         const float *__restrict__ save, int chunk) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = blockIdx.x * 64 + lane;
    const int r0 = blockIdx.y * chunk, r1 = min(m, r0 + chunk);
    const size_t p = (size_t)(col < N ? col : N - 1) / PANEL;
    const int j = (col < N ? col : N - 1) % PANEL;
    for (int base = r0; base < r1; base += 64) {
        const int f = base + lane < r1 ? flags[base + lane] : 0;
        uint64_t mask = __ballot(f != 0);
        for (int nth = 0; mask; nth++, mask &= mask - 1) {
            if ((nth & 3) != wave) continue;
            const int row = base + __builtin_ctzll(mask);
            if (col >= N) continue;
            const float *ar = a + (size_t)row * lda;
            float acc = 0.0f;
            for (int i = 0; i < k; i++)
                acc = __builtin_fmaf(ar[i], widen_one(wv, scales, prec, k, ps, bs, p, j, i), acc);
            const float old = accumulate ? save[(size_t)row * N + col] : 0.0f;
            c[(size_t)row * ldc + col] = epilogue_vals(acc, bias != nullptr, bias ? bias[col] : 0.0f, act, escale,
                                                       accumulate != 0, old);
        }
    }
}

// ---------------------------------------------------------------------------- on the matrix cores
//
// v_mfma_f32_16x16x4_f32 adds its four products one after another, each a fused multiply-add with
// one rounding, subnormals kept: a chain of it over k is bit for bit the reference's fused sum in
// input order (checked against fmaf over wide exponents, subnormal inputs and products, signed
// zeros and infinities). So the exact products run on the matrix cores. Before, a lane summed one
// output and loaded and widened a weight for every multiply-add: 750 x 1024 -> 4096 -> 1024 with
// f16 weights 4474 us, here 115 (110 TFLOP/s); 93 rows of it with int8 weights 1394 and 44 us; the 16
// attention products and the softmax of 375 frames 972 and 160 us, most of it launches.
//
// The bound is the f32 matrix rate: an MFMA keeps its SIMD 32 cycles (a chain of dependent ones
// too), and it runs on the vector ALU's multipliers, so every vector instruction beside it adds its
// own four cycles and each change from vector instructions back to MFMAs about ten more (measured:
// 14.4 ns per MFMA alone, 19.7 with one vector instruction before each, 24.6 with four); LDS reads,
// copies and scalar instructions between MFMAs are free. Hence:
//   - four wavefronts share 16 RB rows, each with a panel of its own: a weight is widened once per
//     RB MFMAs, and the widenings of half a stage (32 inputs) stand together before its MFMAs;
//   - operands come through a ring of NS stages of 64 inputs in LDS, copied straight from global
//     memory (16 bytes per lane, or 4 where rows are not 16-byte aligned or the stage is the ragged
//     last one), and half a stage is read from LDS between the MFMAs of the half before.
// LDS layouts without bank conflicts and with fixed offsets between a lane's reads:
//   A: rows in groups of four, 64 floats each and 64 bytes between groups; chunk c (inputs 4 c ..) of
//      row r at chunk c ^ (r % 4), so four lane addresses reach every input;
//   B: as in the panel (f32 and 16 bits: an MFMA step's 64 values are consecutive; int8: a lane's 16
//      inputs of an output, read a byte per step).
// The weights are the first MFMA operand, so a lane's four sums are consecutive columns of one row.
//
// The last stage's inputs past k enter as (-0) * (+0): adding -0 changes no sum, not even a -0.

constexpr int EXACT_THREADS = 256;
constexpr size_t GFX950_CUS = 256;  // compute units of an MI355X

__device__ __forceinline__ uint32_t lds_address(const void *p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)p;
}
// A wave-uniform address in scalar registers.
__device__ __forceinline__ const void *scalar(const void *p) {
    const uint64_t u = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
    return reinterpret_cast<const void *>(((uint64_t)hi << 32) | lo);
}
// Each lane's 16 (or 4) bytes to LDS at lds + 16 (4) * lane, lds wave-uniform: from base + voff (a
// wave-uniform base, the lane's byte offset) or from the lane's address. A copy reads M0 without an
// interlock, one wait state after a scalar write, and the base's scalar registers five after a vector
// one: scalar()'s v_readfirstlane, or the v_readlane of a spilled register. The compiler adds no wait
// states inside an asm text, so the texts hold them (s_mov counts as one of the five).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void copy16(const void *base, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(scalar(base)) : "memory", "m0");
}
__device__ __forceinline__ void copy4(const void *base, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(voff), "s"(scalar(base)) : "memory", "m0");
}
__device__ __forceinline__ void copy4_lanes(const void *p, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds), "v"(p) : "memory", "m0");
}
#pragma clang diagnostic pop
// Waits until at most `ahead` stages of CPW copies are on the way (ahead <= A). Waiting for fewer
// than are there is safe, so counts beyond vmcnt's 6 bits are cut to 63, and a stage of more copies
// than CPW (the ragged last one) only waits longer.
template <int CPW, int A>
__device__ __forceinline__ void wait_ahead(int ahead) {
    constexpr int N = A * CPW < 63 ? A * CPW : 63;
    if constexpr (A == 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
        if (ahead >= A) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
        else wait_ahead<CPW, A - 1>(ahead);
    }
}

struct ExactArgs {
    const float *a;
    size_t lda;
    int M, K;
    const uint8_t *b;  // the weights' values, or the row-major matrix
    size_t pstride;    // f32: floats between panels; int8, Q8_0: bytes between panels
    size_t istride;    // f32: floats between inputs; int8, Q8_0: bytes between k-blocks
    const float *scales;
    int N, P;  // outputs, panels of 16
    float *c;
    size_t ldc;
    EpiArgs epi;
    int grid_n;  // tiles across the outputs
    int vec;     // outputs are 16-byte aligned and rows hold whole runs of four
};

// The epilogue and stores of RB blocks of 16 rows from m0 on and one panel: lane (lg, lj) holds columns
// 4 lg + 0..3 of row lj of each block.
template <int RB>
__device__ __forceinline__ void store_blocks(const ExactArgs &g, const v4f (&acc)[RB], int m0, int panel, int lg, int lj) {
    const bool has_bias = g.epi.bias != nullptr, accumulate = g.epi.accumulate != 0;
    const int col = panel * PANEL + 4 * lg;
    if (col >= g.N) return;
    float bias[4];
#pragma unroll
    for (int v = 0; v < 4; v++) bias[v] = has_bias && col + v < g.N ? g.epi.bias[col + v] : 0.0f;
#pragma unroll
    for (int r = 0; r < RB; r++) {
        const int row = m0 + r * 16 + lj;
        if (row >= g.M) continue;
        float *cp = g.c + (size_t)row * g.ldc + col;
        if (g.vec) {
            v4f old = {0.0f, 0.0f, 0.0f, 0.0f}, y;
            if (accumulate) old = *reinterpret_cast<const v4f *>(cp);
#pragma unroll
            for (int v = 0; v < 4; v++)
                y[v] = epilogue_vals(acc[r][v], has_bias, bias[v], g.epi.act, g.epi.scale, accumulate, old[v]);
            *reinterpret_cast<v4f *>(cp) = y;
        } else {
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (col + v < g.N)
                    cp[v] = epilogue_vals(acc[r][v], has_bias, bias[v], g.epi.act, g.epi.scale, accumulate,
                                          accumulate ? cp[v] : 0.0f);
        }
    }
}

// PREC: the right-hand side's precision. AW, BW: A rows / the f32 right-hand side take 16-byte copies.
template <uint32_t PREC, int RB, int NS, bool AW, bool BW>
__global__ __launch_bounds__(EXACT_THREADS) void exact_kernel(ExactArgs g) {
    constexpr int KT = 64, TN = 4;  // inputs per stage, panels per workgroup (one per wavefront)
    constexpr bool I8 = PREC == INT8 || PREC == Q8_0, H16 = PREC == F16 || PREC == BF16, RAW = I8 || H16;
    constexpr int AGROUP = 1024 + 64;                  // four rows and the gap after them
    constexpr int PB = I8 ? 1024 : H16 ? 2048 : 4096;  // bytes per panel and stage
    constexpr int ABYTES = 4 * RB * AGROUP, BBYTES = TN * PB, SBYTES = PREC == Q8_0 ? TN * 256 : 0;
    constexpr int STAGE = ABYTES + BBYTES + SBYTES;
    // Copies per wavefront and stage: A's split over the four, the wavefront's own panel (and scales).
    constexpr int ACW = AW ? RB : 4 * RB, BCW = I8 ? 1 : H16 ? 2 : BW ? 4 : 16, SCW = PREC == Q8_0 ? 1 : 0;
    constexpr int CPW = ACW + BCW + SCW;
    static_assert(NS >= 3, "a stage lands while one is multiplied and another's buffer refills");
    __shared__ __attribute__((aligned(16))) uint8_t smem[NS * STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lg = lane >> 4, lj = lane & 15;
    // Contiguous runs of tiles, row by row, per XCD (workgroup L runs on XCD L % 8).
    int L = blockIdx.x;
    const int full = (int)gridDim.x - (int)gridDim.x % 8;
    if (L < full) L = (L % 8) * (full / 8) + L / 8;
    const int by = L / g.grid_n, bx = L % g.grid_n;
    const int m0 = by * RB * 16, panel = bx * TN + wave;
    const size_t p = (size_t)min(panel, g.P - 1);  // a panel past the edge repeats the last, never stored
    const int K = g.K, KB = K / KT + (K % KT != 0);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(smem));
    const float *a0 = g.a + (size_t)m0 * g.lda;

    // Row r (rows past the edge repeat the last) of the tile, from the tile's first row.
    auto row_at = [&](int r) { return (size_t)min(r, g.M - 1 - m0) * g.lda; };
    uint32_t aoff[AW ? RB : 1];
    if constexpr (AW) {
#pragma unroll
        for (int i = 0; i < RB; i++)
            aoff[i] = (uint32_t)(row_at(4 * (wave + 4 * i) + lg) + 4 * (lj ^ lg)) * 4;
    }
    // One row of stage t per copy, the inputs past the last one (t may be the ragged stage) repeating it.
    auto copy_row = [&](int buf, int t, int i, bool ragged) {
        const int r = wave + 4 * i, o = 4 * ((lane >> 2) ^ (r & 3)) + (lane & 3);
        const int in = ragged ? min(o, K - 1 - t * KT) : o;
        copy4_lanes(a0 + row_at(r) + (size_t)t * KT + in, lds0 + buf * STAGE + (r >> 2) * AGROUP + (r & 3) * 256);
    };
    auto copy_b = [&](int buf, int t, int i, bool ragged) {
        const uint32_t sb = lds0 + buf * STAGE + ABYTES + wave * PB;
        const int last = K - 1 - t * KT;
        if constexpr (I8) {
            copy16(g.b + p * g.pstride + (size_t)t * g.istride, lane * 16, sb);
        } else if constexpr (H16) {
            int k = 32 * i + (lane >> 1);
            if (ragged) k = min(k, last);
            copy16(g.b + (p * K + (size_t)t * KT) * PANEL * 2, (uint32_t)(k * PANEL + 8 * (lane & 1)) * 2, sb + i * 1024);
        } else {
            const float *base = reinterpret_cast<const float *>(g.b) + p * g.pstride + (size_t)t * KT * g.istride;
            if constexpr (BW) {
                int k = 16 * i + (lane >> 2);
                if (ragged) k = min(k, last);
                copy16(base, ((uint32_t)k * (uint32_t)g.istride + 4 * (lane & 3)) * 4, sb + i * 1024);
            } else {
                int k = 4 * i + lg;
                if (ragged) k = min(k, last);
                copy4_lanes(base + (size_t)k * g.istride + lj, sb + i * 256);
            }
        }
    };
    auto copy_scales = [&](int buf, int t) {
        const int blocks = (K + Q8_BLOCK - 1) / Q8_BLOCK, b = 2 * t + (lg & 1);
        copy4(g.scales + p * blocks * PANEL, (uint32_t)(min(b, blocks - 1) * PANEL + lj) * 4,
              lds0 + buf * STAGE + ABYTES + BBYTES + wave * 256);
    };
    // Copy i of this wavefront's CPW of a whole stage.
    auto copy_whole = [&](int buf, int t, int i) {
        if (i < ACW) {
            if constexpr (AW) copy16(a0 + (size_t)t * KT, aoff[AW ? i : 0], lds0 + buf * STAGE + (wave + 4 * i) * AGROUP);
            else copy_row(buf, t, i, false);
        } else if (i < ACW + BCW) {
            copy_b(buf, t, i - ACW, false);
        } else if (i < CPW) {
            copy_scales(buf, t);
        }
    };
    auto issue = [&](int buf, int t) {
        if (K - t * KT >= KT) {
#pragma unroll
            for (int i = 0; i < CPW; i++) copy_whole(buf, t, i);
        } else {
#pragma unroll
            for (int i = 0; i < 4 * RB; i++) copy_row(buf, t, i, true);
#pragma unroll
            for (int i = 0; i < BCW; i++) copy_b(buf, t, i, true);
            if constexpr (PREC == Q8_0) copy_scales(buf, t);
        }
    };

    // Half a stage, h (inputs 32 h ..) of buffer buf: step s takes inputs 4 s + lg of row lj (a) and of
    // output lj (w, widened from raw). Pieces 0..7 of its reads are the steps' weights, the others the
    // rows' steps, block by block.
    struct Frags {
        float a[RB][8], w[8];
    };
    int raw[8];
    float rawscale = 0.0f;
    int abase[4];
#pragma unroll
    for (int v = 0; v < 4; v++) abase[v] = (lj >> 2) * AGROUP + (lj & 3) * 256 + ((v ^ (lj & 3)) * 16) + lg * 4;
    const int bbase = ABYTES + wave * PB + (I8 ? lj * 16 + lg : H16 ? lane * 2 : lane * 4);
    constexpr int PIECES = 8 + 8 * RB;
    auto read_piece = [&](int buf, int h, int piece, Frags &f) {
        const uint8_t *st = smem + buf * STAGE;
        if (piece < 8) {
            const int s = piece;
            if constexpr (I8) {
                raw[s] = *reinterpret_cast<const int8_t *>(st + bbase + (2 * h + s / 4) * 256 + 4 * (s % 4));
                if constexpr (PREC == Q8_0)
                    if (s == 0)
                        rawscale = *reinterpret_cast<const float *>(st + ABYTES + BBYTES + wave * 256 + h * 64 + lj * 4);
            } else if constexpr (H16) {
                raw[s] = *reinterpret_cast<const uint16_t *>(st + bbase + (8 * h + s) * 128);
            } else {
                f.w[s] = *reinterpret_cast<const float *>(st + bbase + (8 * h + s) * 256);
            }
        } else {
            const int s = (piece - 8) / RB, r = (piece - 8) % RB, ss = 8 * h + s;
            f.a[r][s] = *reinterpret_cast<const float *>(st + abase[ss % 4] + (ss / 4) * 64 + r * 4 * AGROUP);
        }
    };
    auto read = [&](int buf, int h, Frags &f) {
#pragma unroll
        for (int i = 0; i < PIECES; i++) read_piece(buf, h, i, f);
    };
    float scale = 0.0f;
    if constexpr (PREC == INT8) {
        scale = g.scales[p * PANEL + lj];
        asm volatile("" : "+v"(scale));  // waited for here: in the loop the wait would be for every copy on the way
    }
    auto widen = [&](Frags &f) {
        if constexpr (RAW) {
#pragma unroll
            for (int s = 0; s < 8; s++) {
                if constexpr (I8) f.w[s] = (float)raw[s] * (PREC == INT8 ? scale : rawscale);
                else if constexpr (PREC == F16) f.w[s] = (float)__builtin_bit_cast(_Float16, (uint16_t)raw[s]);
                else f.w[s] = __uint_as_float((uint32_t)raw[s] << 16);
            }
        }
    };
    v4f acc[RB];
#pragma unroll
    for (int r = 0; r < RB; r++) acc[r] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    auto mfma = [&](float w, float a, int r) {
        acc[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, a, acc[r], 0, 0, 0);
    };
    // The half stage's first `left` inputs only.
    auto mma_ragged = [&](const Frags &f, int left) {
#pragma unroll
        for (int s = 0; s < 8; s++) {
            if (4 * s >= left) break;
            const bool in = 4 * s + lg < left;
#pragma unroll
            for (int r = 0; r < RB; r++) mfma(in ? f.w[s] : 0.0f, in ? f.a[r][s] : -0.0f, r);
        }
    };

    // Stage t sits in buffer t % NS. Its second half is read under its first half's MFMAs, and the
    // next stage's first half under its second's, after a barrier that also frees stage t - 1's buffer,
    // which stage t + NS - 1's copies then refill. The main loop takes NS stages at a time while none of
    // the stages it copies is ragged or past the last, so it holds no branch, fixed offsets and fixed waits.
    Frags f0, f1;
#pragma unroll
    for (int s = 0; s < NS - 1; s++)
        if (s < KB) issue(s, s);
    if (KB > 0) {
        wait_ahead<CPW, NS - 2>(min(NS - 2, KB - 1));
        __syncthreads();
        read(0, 0, f0);
    }
    int t = 0, buf = 0, nxt = 1, prev = NS - 1;
    auto advance = [&]() {
        t++;
        prev = buf;
        buf = nxt;
        nxt = nxt + 1 == NS ? 0 : nxt + 1;
    };
    // The eight steps of f, the reads of the half stage (rbuf, rh) into fr spread over the four steps
    // from `first` on, `after(s)` at the end of step s.
    auto half = [&](const Frags &f, int rbuf, int rh, Frags &fr, int first, auto after) {
        constexpr int slots = 4 * RB;
#pragma unroll
        for (int s = 0; s < 8; s++) {
#pragma unroll
            for (int r = 0; r < RB; r++) {
                mfma(f.w[s], f.a[r][s], r);
                const int i = (s - first) * RB + r;
                if (i >= 0 && i < slots) {
#pragma unroll
                    for (int q = PIECES * i / slots; q < PIECES * (i + 1) / slots; q++) read_piece(rbuf, rh, q, fr);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            after(s);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    constexpr int SPREAD = (CPW + 6) / 7;  // copies after each step of the second half but the first
    for (const int main = K / KT - (NS - 1); t + NS <= main; t += NS) {
#pragma unroll
        for (int u = 0; u < NS; u++) {  // the buffers' offsets are constants
            widen(f0);
            __builtin_amdgcn_sched_barrier(0);
            half(f0, u, 1, f1, 0, [](int) {});
            widen(f1);
            __builtin_amdgcn_sched_barrier(0);
            half(f1, (u + 1) % NS, 0, f0, 1, [&](int s) {
                if (s == 0) {
                    wait_ahead<CPW, NS - 3>(NS - 3);
                    __syncthreads();
                } else {
#pragma unroll
                    for (int i = (s - 1) * SPREAD; i < s * SPREAD; i++) copy_whole((u + NS - 1) % NS, t + u + NS - 1, i);
                }
            });
        }
    }
    for (; t < KB; advance()) {
        const int left = K - t * KT;
        const bool more = t + 1 < KB;  // then this stage is whole
        widen(f0);
        if (left >= 32) {
            half(f0, buf, 1, f1, 0, [](int) {});
        } else {
            mma_ragged(f0, left);
            break;
        }
        if (more) {
            wait_ahead<CPW, NS - 3>(min(NS - 3, KB - 2 - t));
            __syncthreads();
            if (t + NS - 1 < KB) issue(prev, t + NS - 1);
        }
        widen(f1);
        if (left >= KT) half(f1, more ? nxt : buf, 0, f0, 0, [](int) {});  // the last one's reads are of no use
        else mma_ragged(f1, left - 32);
    }

    store_blocks<RB>(g, acc, m0, panel, lg, lj);
}

// Sums of few inputs, without the ring: a wavefront takes 16 RB rows of one panel and loads its operands
// in the MFMAs' layout straight from memory, four steps at a time, so no workgroup holds LDS or waits at a
// barrier. Such products are bound by their stores and by how many workgroups are under way, and with the
// ring's LDS one or two fit on a CU. us, 100,000 rows by 64 outputs with the ring / here, f32: 1 input
// 46.5 / 10.1, 16 inputs 48.3 / 19.9, 32 inputs 50.6 / 31.8; f16: 1 input 21.2 / 10.5, 16 inputs 22.3 / 19.6, 24
// inputs 22.9 / 26.8. 10,000 rows by 1024: f32, 32 inputs 48.6 / 43.9, 48 inputs 52.4 / 60.1; int8, 16 inputs
// 28.1 / 27.5, 24 inputs 29.8 / 38.0. Hence the most inputs that it takes; the ring's four wavefronts
// share the rows, which longer sums read often.
template <uint32_t PREC>
constexpr int SHORT = PREC == F32 ? 32 : 16;
template <uint32_t PREC, int RB>
__global__ __launch_bounds__(EXACT_THREADS) void exact_short_kernel(ExactArgs g) {
    const int lane = threadIdx.x & 63, lg = lane >> 4, lj = lane & 15;
    const int tile = blockIdx.x * (EXACT_THREADS / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int panel = tile % g.P, m0 = tile / g.P * RB * 16;
    if (m0 >= g.M) return;
    const float *row[RB];
#pragma unroll
    for (int r = 0; r < RB; r++) row[r] = g.a + (size_t)min(m0 + r * 16 + lj, g.M - 1) * g.lda;
    v4f acc[RB];
#pragma unroll
    for (int r = 0; r < RB; r++) acc[r] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    for (int i0 = 0; i0 < g.K; i0 += 16) {
        float w[4], a[RB][4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int i = i0 + 4 * s + lg, in = min(i, g.K - 1);
            float v;
            if constexpr (PREC == F32)
                v = reinterpret_cast<const float *>(g.b)[(size_t)panel * g.pstride + (size_t)in * g.istride + lj];
            else
                v = widen_one(g.b, g.scales, PREC, g.K, g.pstride, g.istride, panel, lj, in);
            w[s] = i < g.K ? v : 0.0f;
#pragma unroll
            for (int r = 0; r < RB; r++) a[r][s] = i < g.K ? row[r][in] : -0.0f;
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (i0 + 4 * s >= g.K) break;
#pragma unroll
            for (int r = 0; r < RB; r++) acc[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s], a[r][s], acc[r], 0, 0, 0);
        }
    }
    store_blocks<RB>(g, acc, m0, panel, lg, lj);
}

// launch(g) for runs of rows, whole blocks of `rows` of them: about RUN_GROUPS workgroups each, since HIP
// cuts the number of threads to 32 bits without an error: 2^30 + 70 rows by one panel in one launch left
// all but the first rows as they were. A run takes milliseconds.
constexpr size_t RUN_GROUPS = (size_t)1 << 20;
template <class F>
hipError_t launch_runs(ExactArgs g, size_t groups_per_block, size_t rows, F launch) {
    if (groups_per_block * EXACT_THREADS > (size_t)UINT32_MAX) return hipErrorInvalidValue;
    const float *a = g.a;
    float *c = g.c;
    const size_t m = (size_t)g.M, run = std::max<size_t>(1, RUN_GROUPS / groups_per_block) * rows;
    for (size_t m0 = 0; m0 < m; m0 += run) {
        g.a = a + m0 * g.lda;
        g.c = c + m0 * g.ldc;
        g.M = (int)std::min(run, m - m0);
        launch(g);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <uint32_t PREC, int RB, int NS>
hipError_t launch_tiles(ExactArgs g, bool aw, bool bw, hipStream_t s) {
    g.grid_n = (int)div_ceil((size_t)g.P, (size_t)4);
    auto kernel = aw ? &exact_kernel<PREC, RB, NS, true, true> : &exact_kernel<PREC, RB, NS, false, true>;
    if constexpr (PREC == F32) {
        if (!bw) kernel = aw ? &exact_kernel<PREC, RB, NS, true, false> : &exact_kernel<PREC, RB, NS, false, false>;
    }
    return launch_runs(g, (size_t)g.grid_n, RB * 16, [&](const ExactArgs &r) {
        const size_t tiles = (size_t)r.grid_n * div_ceil((size_t)r.M, (size_t)(RB * 16));
        hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(EXACT_THREADS), 0, s, r);
    });
}

template <uint32_t PREC, int RB>
hipError_t launch_short(const ExactArgs &g, hipStream_t s) {
    constexpr size_t WAVES = EXACT_THREADS / 64;
    return launch_runs(g, div_ceil((size_t)g.P, WAVES), RB * 16, [&](const ExactArgs &r) {
        const size_t tiles = (size_t)r.P * div_ceil((size_t)r.M, (size_t)(RB * 16));
        hipLaunchKernelGGL(HIP_KERNEL_NAME(exact_short_kernel<PREC, RB>), dim3((unsigned)div_ceil(tiles, WAVES)),
                           dim3(EXACT_THREADS), 0, s, r);
    });
}

template <uint32_t PREC>
hipError_t launch_exact_as(ExactArgs g, hipStream_t s) {
    // 16-byte copies of rows that are 16 bytes aligned; their lane offsets are 32-bit over 64 rows.
    const bool aw = reinterpret_cast<uintptr_t>(g.a) % 16 == 0 && g.lda % 4 == 0 && g.lda < ((size_t)1 << 24);
    const bool bw = reinterpret_cast<uintptr_t>(g.b) % 16 == 0 && g.istride % 4 == 0 && g.istride < ((size_t)1 << 24);
    g.vec = ((reinterpret_cast<uintptr_t>(g.c) | g.ldc * sizeof(float)) % 16) == 0 && g.N % 4 == 0;
    // Few inputs: four row blocks per wavefront where that leaves sixteen wavefronts per CU.
    if (g.K <= SHORT<PREC>)
        return (size_t)g.P * g.M >= (size_t)64 * GFX950_CUS * 16 ? launch_short<PREC, 4>(g, s) : launch_short<PREC, 1>(g, s);
    // Row blocks per workgroup: the fewest row blocks on the busiest CU (workgroups per CU, rounded up,
    // times RB), and of equals the largest, whose widenings serve more MFMAs. us, f16, RB = 1 / 2 / 3 /
    // 4: 93 x 4096 -> 1024 24.2 / 39.6 / 53.5 / 69.2; 375 x 4096 -> 1024 43.6 / 42.6 / 56.7 / 71.4;
    // 750 x 4096 -> 1024 65.7 / 76.6 / 62.4 / 80.6; 1000 x 4096 -> 1024 85.9 / 83.0 / 114.8 / 78.5.
    // The largest loss against the best of the four there and at 1024 -> 4096 is 9%.
    size_t best = 0, least = SIZE_MAX;
    for (size_t rb = 1; rb <= 4; rb++) {
        const size_t tiles = div_ceil((size_t)g.M, 16 * rb) * div_ceil((size_t)g.P, 4);
        const size_t load = div_ceil(tiles, GFX950_CUS) * rb;
        if (load <= least) {
            least = load;
            best = rb;
        }
    }
    switch (best) {
    case 1: return launch_tiles<PREC, 1, 4>(g, aw, bw, s);
    case 2: return launch_tiles<PREC, 2, 3>(g, aw, bw, s);
    case 3: return launch_tiles<PREC, 3, 3>(g, aw, bw, s);
    default: return launch_tiles<PREC, 4, 3>(g, aw, bw, s);
    }
}

}  // namespace

hipError_t launch_rowmajor(const float *a, size_t lda, size_t m, size_t k, const float *b, size_t ldb, size_t n,
                           float *c, size_t ldc, const EpiArgs &epi, hipStream_t s) {
    if (m == 0 || n == 0) return hipSuccess;
    // The view's panels are 16 columns apart and hold whole rows of 16 (the caller's check), as the
    // packed panels are: only the strides differ.
    return launch_exact_as<F32>(ExactArgs{a, lda, (int)m, (int)k, reinterpret_cast<const uint8_t *>(b), PANEL, ldb,
                                          nullptr, (int)n, (int)div_ceil(n, (size_t)PANEL), c, ldc, epi, 0, 0},
                                s);
}

hipError_t launch_exact(const float *a, size_t lda, size_t m, const DeviceWeights &w, float *c, size_t ldc,
                        const EpiArgs &epi, hipStream_t s) {
    if (m == 0 || w.n == 0) return hipSuccess;
    ExactArgs g{a, lda, (int)m, (int)w.k, w.values, w.panel_stride, w.blk_stride, w.scales, (int)w.n, (int)w.panels,
                c, ldc, epi, 0, 0};
    switch (w.precision) {
    case F32:
        g.pstride = w.k * PANEL;
        g.istride = PANEL;
        return launch_exact_as<F32>(g, s);
    case F16: return launch_exact_as<F16>(g, s);
    case BF16: return launch_exact_as<BF16>(g, s);
    case INT8: return launch_exact_as<INT8>(g, s);
    default: return launch_exact_as<Q8_0>(g, s);
    }
}

hipError_t launch_exact_rows(const float *a, size_t lda, size_t m, const DeviceWeights &w, float *c, size_t ldc,
                             const EpiArgs &epi, const int32_t *flags, const float *save, hipStream_t s) {
    if (m == 0 || w.n == 0) return hipSuccess;
    // About 2048 workgroups: the column groups times row chunks of whole groups of 64 rows.
    const size_t cols = div_ceil(w.n, 64), groups = div_ceil(m, 64);
    size_t chunks = 2048 / cols;
    chunks = chunks < 1 ? 1 : (chunks > groups ? groups : chunks);
    const size_t chunk = div_ceil(groups, chunks) * 64;
    dim3 grid((unsigned)cols, (unsigned)div_ceil(m, chunk));
    hipLaunchKernelGGL(exact_rows_kernel, grid, dim3(256), 0, s, a, lda, (int)m, (int)w.k, w.values, w.scales,
                       w.precision, (int)w.n, w.panel_stride, w.blk_stride, c, ldc, epi.bias, epi.act, epi.scale,
                       epi.accumulate, flags, save, (int)chunk);
    return hipGetLastError();
}

}  // namespace tg
