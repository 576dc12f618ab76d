// Prefill / vision GEMM on CDNA4 matrix cores:
//   C[b][m][n] = sum_k A[b][m][k] * B[b][n][k]     (NT: both operands K-contiguous)
// A and B fp16 or bf16, fp32 accumulation, C stored fp32 / fp16 / bf16.
//
// Replaces gemm_image (src/kernels/gemm.cl:157-200) as the prefill path
// (dispatch_gemm_image, src/engine/compute.cpp:90-120; every projection in
// src/models/moondream2.cpp:374-508) and serves the batched attention scores
// Q*K^T (the dot of src/kernels/attention.cl:84-88).
//
// Structure.  A block of WGM x WGN waves owns a BM x BN tile of C; each wave a
// (BM/WGM) x (BN/WGN) sub-tile of 32x32 v_mfma_f32_32x32x16 tiles.
// K advances in 64-wide stages held in an LDS ring of STAGES slots:
//  * global -> LDS with direct 16-byte loads (global_load_lds_dwordx4): one
//    wave instruction moves 8 rows x 128 bytes (a 64-element K slice of 8
//    rows) straight into LDS, no registers involved, so up to STAGES-1 stages
//    are in flight while the MFMAs work on the oldest;
//  * LDS rows are 128 bytes; the 16-byte slot s of row r is stored at slot
//    s ^ ((r >> 1) & 7).  gfx950's LDS serves a ds_read_b128 16 lanes at a
//    time from 64 four-byte banks (a 256-byte period, two rows), so the 16
//    rows read by one phase must occupy 16 distinct (row parity, slot) pairs;
//    an (r & 7) swizzle leaves rows r and r+8 on the same banks (measured:
//    half of all LDS cycles were bank conflicts).  The swizzle is applied on
//    the global side: lane i of a load instruction writes LDS bytes
//    [16i, 16i+16) of its 8-row group g and so fetches logical slot
//    (i & 7) ^ ((4g + (i >> 4)) & 7);
//  * one barrier per stage: after it, the slot computed in the previous
//    iteration is refilled.
// That is the kernel of the small tiles (gemm_mfma_kernel); tiles from 128 x
// 128 up share its layouts but alternate two groups of waves
// (gemm_pingpong_kernel).
// Rows beyond M / N are clamped to the last valid row (their products land in
// outputs that are never stored).  K beyond the operand's readable width is
// zero-filled by a guarded load path used only for the last stage.
// Operand layout of v_mfma_f32_32x32x16_{f16,bf16}: lane l supplies
// A[l%32][8*(l/32) .. +7] and B^T[l%32][8*(l/32) .. +7]; accumulator register
// r of lane l is C[8*(r/4) + 4*(l/32) + r%4][l%32].
#include "common.h"
#include "device_math.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>

namespace mvlm {

// LDS geometry of a stage BK elements wide: one row per operand row, RB bytes
// (LPR 16-byte slots); one direct-load instruction fills RPI rows (1 KiB).
// Slot s of row r is stored at s ^ swz(r): a ds_read_b128 phase (16 lanes,
// 16 consecutive rows, one logical slot) then hits 16 distinct 16-byte bank
// groups of the 256-byte bank period (one 256-byte row, two 128-byte rows, or
// four 64-byte rows).
template <int BK>
struct StageGeom {
    static_assert(BK == 32 || BK == 64 || BK == 128, "stage width");
    static constexpr int ROWH = BK, RB = 2 * BK, LPR = RB / 16, RPI = 1024 / RB;
    __device__ static __forceinline__ int swz(int r) {
        return BK == 128 ? r & 15 : BK == 64 ? (r >> 1) & 7 : (r >> 2) & 3;
    }
};

struct GemmArgs {
    const uint16_t* A;
    const uint16_t* B;
    void* C;
    int c_dtype;
    int M, N, K;
    int64_t lda, ldb, ldc, sA, sB, sC;
    int kread_b;        // B rows are readable (zero padded) up to this K (>= K)
    int tiles_m, tiles_n;
    Epilogue ep;        // applied when ep_on (mul / res indexed like C)
    int ep_on;
    // split-K: grid z = batch * splits; split s covers K stages
    // [s * split_stages, (s + 1) * split_stages) and, when splits > 1, writes
    // its fp32 partial to ws[(b * splits + s) * M * N + m * N + n] for
    // gemm_splitk_reduce_kernel (which then applies the epilogue)
    int splits, split_stages;
    float* ws;
    // 4 consecutive columns of a row start 16-byte (fp32) / 8-byte (16-bit)
    // aligned in C (vec_c) and in the split partials (vec_ws), so one vector
    // store writes them
    int vec_c, vec_ws;
    // the epilogue's operands too, and N % 4 == 0: they are read four at a time
    int vec_ep;
};

// fp32 partial of 4 consecutive columns (n_left of them below N; the row
// starts 16-byte aligned)
__device__ __forceinline__ void store_partial4(float* ws, int64_t i, f32x4 v, int n_left) {
    if (n_left >= 4) {
        asm_global_store_b128_wt(ws + i, __builtin_bit_cast(u32x4, v));
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (e < n_left) ws[i + e] = v[e];
}

// Four consecutive epilogue operands (16-byte / 8-byte aligned), as stored and
// widened.
__device__ __forceinline__ u32x4 load_operand4(const void* base, int64_t i, int dtype) {
    if (dtype == 0) return *reinterpret_cast<const u32x4*>((const float*)base + i);
    const u32x2 h = *reinterpret_cast<const u32x2*>((const uint16_t*)base + i);
    return u32x4{h[0], h[1], 0, 0};
}
__device__ __forceinline__ f32x4 widen_operand4(u32x4 r, int dtype) {
    if (dtype == 0) return __builtin_bit_cast(f32x4, r);
    const uint16_t h[4] = {(uint16_t)r[0], (uint16_t)(r[0] >> 16), (uint16_t)r[1], (uint16_t)(r[1] >> 16)};
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = dtype == 1 ? f16_bits_to_f32(h[e]) : bf16_bits_to_f32(h[e]);
    return v;
}
__device__ __forceinline__ float widen_operand(uint32_t r, int dtype) {
    return dtype == 0 ? __uint_as_float(r) : dtype == 1 ? f16_bits_to_f32((uint16_t)r) : bf16_bits_to_f32((uint16_t)r);
}
// apply_epilogue's two halves on four consecutive columns, the operands loaded
// before: act(v + bias), then * mul + res
__device__ __forceinline__ f32x4 activate4(const Epilogue& e, f32x4 v, u32x4 bias) {
    if (e.bias) v += widen_operand4(bias, e.dtype);
    if (e.act == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = gelu_tanh(v[i]);
    } else if (e.act == 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = silu(v[i]);
    }
    return v;
}
__device__ __forceinline__ f32x4 combine4(const Epilogue& e, f32x4 v, u32x4 mul, u32x4 res) {
    if (e.mul) v *= widen_operand4(mul, e.dtype);
    if (e.res) v += widen_operand4(res, e.dtype);
    return v;
}

// C row `row_off` (element offset of the row), columns col..col+3: output dtype,
// one 16- or 8-byte store when the row is aligned for it, written through L2 (C
// is tens of MB at the prefill shapes)
__device__ __forceinline__ void store_c4(const GemmArgs& p, int64_t row_off, int col, f32x4 v) {
    const int n_left = p.N - col;
    if (n_left <= 0) return;
    const int64_t i = row_off + col;
    if (p.vec_c && n_left >= 4) {
        if (p.c_dtype == 0) {
            asm_global_store_b128_wt((float*)p.C + i, __builtin_bit_cast(u32x4, v));
        } else {
            u32x2 h;
            if (p.c_dtype == 1) {
                h[0] = f32_to_f16_bits(v[0]) | ((uint32_t)f32_to_f16_bits(v[1]) << 16);
                h[1] = f32_to_f16_bits(v[2]) | ((uint32_t)f32_to_f16_bits(v[3]) << 16);
            } else {
                h[0] = f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16);
                h[1] = f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16);
            }
            asm_global_store_b64_wt((uint16_t*)p.C + i, h);
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (e < n_left) store_out(p.C, i + e, v[e], p.c_dtype);
}

template <bool BF16>
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
    if constexpr (BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Direct loads of one operand's stage: ROWS rows starting at tile row r0,
// K columns [k0, k0+BK).  Wave w of NW issues RPI-row groups w, w+NW, ...;
// lane i writes LDS bytes [16i, 16i+16) of its group, i.e. row RPI g + i/LPR,
// physical slot i%LPR, and so fetches logical slot (i%LPR) ^ swz(row).
template <int BK, int ROWS, int NW>
__device__ __forceinline__ void stage_direct(const uint16_t* __restrict__ base, int64_t ld, int r0, int rmax, int k0,
                                             uint16_t* lds, int wave, int lane) {
    using G = StageGeom<BK>;
    static_assert((ROWS / G::RPI) % NW == 0, "row groups must split evenly over the waves");
#pragma unroll
    for (int t = 0; t < ROWS / (G::RPI * NW); ++t) {
        const int g = wave + NW * t;
        const int lr = G::RPI * g + lane / G::LPR;
        const int ls = (lane % G::LPR) ^ G::swz(lr);
        const int r = min(r0 + lr, rmax);
        const uint16_t* src = base + (int64_t)r * ld + k0 + ls * 8;
        asm_global_load_lds_b128(src, __builtin_amdgcn_readfirstlane(lds_offset(lds + G::RPI * g * G::ROWH)));
    }
}

// Guarded loads of the last stage: 16-byte chunks at or beyond kread are zero.
template <int BK, int ROWS, int NW>
__device__ __forceinline__ void stage_guarded(const uint16_t* __restrict__ base, int64_t ld, int r0, int rmax, int k0,
                                              int kread, uint16_t* lds, int wave, int lane) {
    using G = StageGeom<BK>;
    static_assert((ROWS / G::RPI) % NW == 0, "row groups must split evenly over the waves");
#pragma unroll
    for (int t = 0; t < ROWS / (G::RPI * NW); ++t) {
        const int g = wave + NW * t;
        const int lr = G::RPI * g + lane / G::LPR;
        const int ls = (lane % G::LPR) ^ G::swz(lr);
        const int r = min(r0 + lr, rmax);
        const int k = k0 + ls * 8;
        u32x4 v = {0, 0, 0, 0};
        if (k < kread) v = *reinterpret_cast<const u32x4*>(base + (int64_t)r * ld + k);
        *reinterpret_cast<u32x4*>(lds + G::RPI * g * G::ROWH + lane * 8) = v;
    }
}

// The wave's TM x TN accumulator tiles to C, with the epilogue (EP) or without,
// or (not EP) to the split partials ws: tile (i, j) has its first element at row
// row_of(i), column col_of(j).  cst: the wave's 32 x CSTAGE floats of LDS
// staging.  EP is a kernel of its own: code that a launch jumps over costs it
// instruction fetches.  With one kernel for both, 64 x 2048 x 64 took 6.0 us (now
// 5.6), 4 x 64 x 320 with bias and GELU 6.7 (5.4), 4096^3 114 (111).
constexpr int CSTAGE = 36;
template <bool EP, int TM, int TN, int GT, typename RowOf, typename ColOf>
__device__ __forceinline__ void store_tiles(const GemmArgs& p, f32x16 (&acc)[TM][TN], float* cst, int64_t c_off,
                                            float* ws, int lane, RowOf row_of, ColOf col_of) {
    if constexpr (!EP) {
        if (!(ws ? p.vec_ws : p.vec_c)) {   // rows off the vector grid: straight from the accumulators, 32 columns per row
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int col = col_of(j) + (lane & 31);
                    if (col >= p.N) continue;
                    auto each_row = [&](auto&& put) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int row = row_of(i) + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                            if (row < p.M) put(row, acc[i][j][r]);
                        }
                    };
                    if (ws) each_row([&](int row, float v) { ws[(int64_t)row * p.N + col] = v; });
                    else each_row([&](int row, float v) { store_out(p.C, c_off + (int64_t)row * p.ldc + col, v, p.c_dtype); });
                }
            return;
        }
    }
    // Aligned rows: through LDS.  Each wave writes one 32x32 accumulator tile
    // at a time into its own region of the (now idle) ring, row-major with a
    // 36-float pitch (rows r and r+4, written by lanes l and l+32, land 16
    // banks apart), and reads it back as 4 consecutive columns per lane, 8 rows
    // per pass: 16-byte global stores, and per-element code (epilogue, dtype)
    // in a loop rather than unrolled over the 16 * TM * TN accumulators.
    constexpr int CS = CSTAGE, T = TM * TN;
    static_assert(T % GT == 0, "whole groups");
    const int srow = lane >> 3, scol = (lane & 7) * 4;
    // passes of 8 rows that a tile whose first row is row0 has inside C
    auto passes = [&](int row0) { return min(4, (p.M - row0 + 7) >> 3); };
    auto stage_tile = [&](f32x16& c) {
#pragma unroll
        for (int r = 0; r < 16; ++r) cst[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * CS + (lane & 31)] = c[r];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave's writes, before its reads
    };
    if constexpr (EP) {
        if (!p.vec_ep) {
            // Rows or operands off the vector grid: element by element, 32
            // columns of two rows at a time, in a loop of four such passes whose
            // operands are requested one round ahead (729 x 3457 x 1152 with bias
            // and residual 33.6 us when each waited for its own).
            const int ecol = lane & 31, erow = lane >> 5;
            __syncthreads();   // every wave is done with the ring (all its loads have landed)
            static_for<T>([&](auto IJ) {
                constexpr int i = decltype(IJ)::value / TN, j = decltype(IJ)::value % TN;
                const int row0 = row_of(i) + erow, col = col_of(j) + ecol, ccol = min(col, p.N - 1);
                const int rounds = passes(row_of(i));
                if (rounds <= 0 || col_of(j) >= p.N) return;
                uint32_t mul[4], res[4];
                auto request = [&](const void* base, int t0, uint32_t (&to)[4]) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const int64_t idx = c_off + (int64_t)min(row0 + 2 * (t0 + t), p.M - 1) * p.ldc + ccol;
                        to[t] = p.ep.dtype == 0 ? ((const uint32_t*)base)[idx] : ((const uint16_t*)base)[idx];
                    }
                };
                if (p.ep.mul) request(p.ep.mul, 0, mul);
                if (p.ep.res) request(p.ep.res, 0, res);
                const float bias = p.ep.bias ? load_as_f32(p.ep.bias, ccol, p.ep.dtype) : 0.0f;
                stage_tile(acc[i][j]);
#pragma unroll 1
                for (int q = 0; q < rounds; ++q) {
                    uint32_t m[4], r[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        m[t] = mul[t];
                        r[t] = res[t];
                    }
                    if (p.ep.mul && q + 1 < rounds) request(p.ep.mul, 4 * q + 4, mul);
                    if (p.ep.res && q + 1 < rounds) request(p.ep.res, 4 * q + 4, res);
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const int row = 8 * q + 2 * t;
                        float x = cst[(row + erow) * CS + ecol] + bias;
                        if (p.ep.act == 1) x = gelu_tanh(x);
                        else if (p.ep.act == 2) x = silu(x);
                        if (p.ep.mul) x *= widen_operand(m[t], p.ep.dtype);
                        if (p.ep.res) x += widen_operand(r[t], p.ep.dtype);
                        if (row0 + row < p.M && col < p.N)
                            store_out(p.C, c_off + (int64_t)(row0 + row) * p.ldc + col, x, p.c_dtype);
                    }
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // reads done before the next tile's writes
            });
            return;
        }
    }
    // The epilogue's operands are requested four columns at a time for GT tiles
    // at once (all of a wave's, but for the 128 accumulators of 256 x 256 and
    // tiles of which two share a CU), before the tiles pass through LDS: one wait
    // for a group's operands and not one per element, which with a tanhf per
    // element made 768 x 8192 x 2048 with bias and GELU take 51 us against 34
    // without; a Phi-1.5 block of 768 rows went 170 -> 153 us, a SigLIP block of
    // 729 101 -> 91.  In-place operands are safe: an element's are read by the
    // thread that later stores it.
    u32x4 bias[TN], mul[GT][4], res[GT][4];
    auto load_group = [&](auto G) {
        auto each = [&](const void* base, u32x4 (&to)[GT][4]) {
            static_for<GT>([&](auto X) {
                constexpr int x = decltype(X)::value, ij = decltype(G)::value * GT + x, i = ij / TN, j = ij % TN;
                const int col = min(col_of(j) + scol, p.N - 4);
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    to[x][t] = load_operand4(base, c_off + (int64_t)min(row_of(i) + srow + 8 * t, p.M - 1) * p.ldc + col,
                                             p.ep.dtype);
            });
        };
        if (p.ep.mul) each(p.ep.mul, mul);
        if (p.ep.res) each(p.ep.res, res);
    };
    if constexpr (EP) {
        if (p.ep.bias)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                bias[j] = load_operand4(p.ep.bias, min(col_of(j) + scol, p.N - 4), p.ep.dtype);
        load_group(std::integral_constant<int, 0>{});
    }
    __syncthreads();   // every wave is done with the ring (all its loads have landed)
    // (compile-time tile indices: a rolled tile loop would index acc at run time
    // and move it to scratch memory)
    static_for<T>([&](auto IJ) {
        constexpr int ij = decltype(IJ)::value, i = ij / TN, j = ij % TN;
        if constexpr (EP && ij > 0 && ij % GT == 0) load_group(std::integral_constant<int, ij / GT>{});
        const int row0 = row_of(i), col = col_of(j) + scol, nt = passes(row0);
        if (nt <= 0 || col_of(j) >= p.N) return;
        stage_tile(acc[i][j]);
        if constexpr (EP) {
            // in a loop and back to LDS: unrolled over every element of the
            // wave this code alone would be tens of KB, run once (the Phi-1.5
            // block: 159 -> 153 us)
            if (p.ep.bias || p.ep.act) {
#pragma unroll 1
                for (int t = 0; t < nt; ++t) {
                    f32x4* v = reinterpret_cast<f32x4*>(cst + (srow + 8 * t) * CS + scol);
                    *v = activate4(p.ep, *v, bias[j]);
                }
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int row = row0 + srow + 8 * t;
                const f32x4 v = combine4(p.ep, *reinterpret_cast<const f32x4*>(cst + (srow + 8 * t) * CS + scol),
                                         mul[ij % GT][t], res[ij % GT][t]);
                if (row < p.M) store_c4(p, c_off + (int64_t)row * p.ldc, col, v);
            }
        } else {
            for (int t = 0; t < nt; ++t) {
                const int row = row0 + srow + 8 * t;
                const f32x4 v = *reinterpret_cast<const f32x4*>(cst + (srow + 8 * t) * CS + scol);
                if (row >= p.M) continue;
                if (ws) store_partial4(ws, (int64_t)row * p.N + col, v, p.N - col);
                else store_c4(p, c_off + (int64_t)row * p.ldc, col, v);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // reads done before the next tile's writes
    });
}

// PER_CU blocks are resident on a CU: the registers of their waves must fit too.
// (128 x 128 with 32-wide stages and the operands of two tiles held at once took
// 132 registers, one block instead of two: 3264 x 20864 x 128 104 us, now 82.)
template <bool BF16, bool EP, int BM, int BN, int BK, int STAGES, int WGM, int WGN, int PER_CU>
__global__ __launch_bounds__(64 * WGM * WGN, PER_CU* WGM* WGN > 8 ? PER_CU * WGM * WGN / 4 : 2) void gemm_mfma_kernel(const GemmArgs p) {
    using G = StageGeom<BK>;
    constexpr int ROWH = G::ROWH;
    constexpr int NW = WGM * WGN;                // waves per block (WGM x WGN grid)
    constexpr int WM = BM / WGM, WN = BN / WGN;  // wave sub-tile
    constexpr int TM = WM / 32, TN = WN / 32;    // 32x32 MFMA tiles per wave
    constexpr int LA = (BM + BN) / G::RPI / NW;  // direct-load instructions per wave per stage
    constexpr int SLOT = (BM + BN) * ROWH;       // elements per ring slot
    static_assert(TM + TN <= 15, "fragment reads must fit the lgkmcnt field");
    // the store pass reuses the ring: a 32 x 36 fp32 staging tile per wave
    static_assert(STAGES * SLOT * 2 >= NW * 32 * CSTAGE * 4, "ring too small for the store staging");
    __shared__ __attribute__((aligned(1024))) uint16_t smem[STAGES * SLOT];

    // Tile order: blocks are dealt round-robin to the 8 XCDs; give each XCD a
    // contiguous run of tiles in which the M tiles of one N tile are adjacent,
    // so the blocks reading the same weight tile share that XCD's L2.
    const int tiles = p.tiles_m * p.tiles_n;
    int t = blockIdx.x;
    const int per = tiles / 8;
    if (t < 8 * per) t = (t % 8) * per + t / 8;
    const int tm = t % p.tiles_m, tn = t / p.tiles_m;
    const int m0 = tm * BM, n0 = tn * BN;

    const int batch = blockIdx.z / p.splits, split = blockIdx.z % p.splits;
    const uint16_t* __restrict__ A = p.A + (int64_t)batch * p.sA;
    const uint16_t* __restrict__ B = p.B + (int64_t)batch * p.sB;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave / WGN, wn = wave % WGN;
    const int K = p.K;
    const int nk_all = (K + BK - 1) / BK;
    const int kt0 = split * p.split_stages;                     // this split's first stage
    const int nk = min(nk_all - kt0, p.split_stages);           // stages of this split (>= 1)
    // the global last stage needs the guarded path when it reaches past K (A)
    // or past B's zero-padded width
    const bool tail_a = (nk_all * BK > K) && kt0 + nk == nk_all;
    const bool tail_b = (nk_all * BK > p.kread_b) && kt0 + nk == nk_all;

    auto issue = [&](int kt) {
        uint16_t* slot = smem + (kt % STAGES) * SLOT;
        const int k0 = (kt0 + kt) * BK;
        const bool last = (kt == nk - 1);
        if (last && tail_a) stage_guarded<BK, BM, NW>(A, p.lda, m0, p.M - 1, k0, K, slot, wave, lane);
        else stage_direct<BK, BM, NW>(A, p.lda, m0, p.M - 1, k0, slot, wave, lane);
        if (last && tail_b)
            stage_guarded<BK, BN, NW>(B, p.ldb, n0, p.N - 1, k0, p.kread_b, slot + BM * ROWH, wave, lane);
        else stage_direct<BK, BN, NW>(B, p.ldb, n0, p.N - 1, k0, slot + BM * ROWH, wave, lane);
    };

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    // Fragment reads of k-step ks of the stage held in ring slot `slot_idx`.
    // They are inline-asm LDS reads with explicit waits (device_math.h): the
    // compiler's own waits would put vmcnt(0) before every read (the ring is
    // filled by direct loads) and merge the loop-carried reads into
    // lgkmcnt(0).  Row r of a fragment is lane&31 plus a multiple of 32, so its
    // swizzle is the lane's; byte offsets: row * RB + slot * 16.
    struct Frags { u32x4 a[TM]; u32x4 b[TN]; };
    const uint32_t lds0 = lds_offset(smem);
    const uint32_t a_lane = (uint32_t)((wm * WM + (lane & 31)) * ROWH * 2);
    const uint32_t b_lane = (uint32_t)((BM + wn * WN + (lane & 31)) * ROWH * 2);
    const int swz = G::swz(lane & 31), half = lane >> 5;
    auto load_frags = [&](int slot_idx, int ks, Frags& f) {
        const uint32_t base = lds0 + (uint32_t)(slot_idx * SLOT * 2) + (uint32_t)((((2 * ks + half) ^ swz)) << 4);
#pragma unroll
        for (int i = 0; i < TM; ++i) f.a[i] = asm_lds_read_b128(base + a_lane + i * 32 * ROWH * 2);
#pragma unroll
        for (int j = 0; j < TN; ++j) f.b[j] = asm_lds_read_b128(base + b_lane + j * 32 * ROWH * 2);
    };
    // wait until at most `newer` LDS reads are pending, then tie f to the wait
    auto ready = [&](Frags& f, bool newer) {
        if (newer) asm_wait_lgkmcnt<TM + TN>();
        else asm_wait_lgkmcnt<0>();
#pragma unroll
        for (int i = 0; i < TM; ++i) asm_pin(f.a[i]);
#pragma unroll
        for (int j = 0; j < TN; ++j) asm_pin(f.b[j]);
    };
    // A wave of one accumulator tile sums its k-steps in four chains, a quarter of
    // the roundings in a row each: K = 2112 against 64 bits 2.75e-7 -> 1.34e-7
    // without a split, 1.36e-7 -> 0.84e-7 with four.  Two chains left 66x5836x1024
    // at 1.28e-7, where more splits had 0.95e-7; 0.94e-7 with four.  The time is
    // one chain's within 1% (32x2048x2048 9.3 us); 122 and 156 registers, as many
    // blocks on a CU.
    constexpr int CHAINS = TM * TN == 1 ? 4 : 1;
    static_assert(BK / 16 % CHAINS == 0, "a k-step's chain is the same in every stage");
    f32x16 chain[CHAINS];                             // chain 0 is acc
#pragma unroll
    for (int c = 1; c < CHAINS; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) chain[c][r] = 0.0f;
    auto mma = [&](const Frags& f, auto KS) {
        constexpr int c = decltype(KS)::value % CHAINS;
        if constexpr (c > 0) {
            chain[c] = mfma32<BF16>(f.a[0], f.b[0], chain[c]);
        } else {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = mfma32<BF16>(f.a[i], f.b[j], acc[i][j]);
        }
    };
    // Stage s has landed in LDS for every wave once this returns.  `later`
    // stages were issued after s; those issued by the direct path may stay in
    // flight (vmcnt counts them in issue order).
    auto wait_stage = [&](int s, int later) {
        const int later_direct = later - ((later > 0 && s + later == nk - 1 && (tail_a || tail_b)) ? 1 : 0);
        if (later_direct >= 2) asm_wait_vmcnt<(2 * LA <= 63) ? 2 * LA : LA>();   // LA: conservative
        else if (later_direct == 1) asm_wait_vmcnt<LA>();
        else asm_wait_vmcnt<0>();
        // A bare s_barrier, not __syncthreads(): the latter's release fence
        // would wait for every in-flight stage (vmcnt(0)).  LDS traffic (this
        // wave's last fragment reads of the slot about to be refilled, and the
        // guarded stage's ds_writes) is drained first.
        asm_wait_lgkmcnt<0>();
        __builtin_amdgcn_s_barrier();
    };

#pragma unroll
    for (int s = 0; s < STAGES; ++s)
        if (s < nk) issue(s);
    wait_stage(0, min(STAGES, nk) - 1);

    // Main loop.  Fragments are double-buffered: the reads of k-step ks+1 are
    // issued before the MFMAs of k-step ks.  Before the last k-step's MFMAs the
    // wave waits for the next stage and meets the others at the barrier, then
    // refills the current slot with stage kt+STAGES (its last reads, k-step 3,
    // were issued during k-step 2 and drained before the barrier) and reads the
    // next stage's first fragments, so neither the barrier nor that read sits
    // in front of an idle matrix core.  Stage kt+1 was issued STAGES-1
    // iterations before it is waited for.
    // Two fragment sets alternate by k-step parity (BK/16 = 4 or 2 k-steps per
    // stage, so a stage always starts on set 0); with the k-step loop unrolled
    // they are distinct registers and no copies are needed.
    Frags f[2];
    load_frags(0, 0, f[0]);
    for (int kt = 0; kt < nk; ++kt) {
        const int slot_idx = kt % STAGES;
        static_for<BK / 16>([&](auto KS) {
            constexpr int ks = decltype(KS)::value;
            Frags& nxt = f[(ks + 1) & 1];
            if (ks < BK / 16 - 1) {
                load_frags(slot_idx, ks + 1, nxt);
            } else if (kt + 1 < nk) {
                wait_stage(kt + 1, min(kt + STAGES - 1, nk - 1) - (kt + 1));
                if (kt + STAGES < nk) issue(kt + STAGES);
                load_frags((kt + 1) % STAGES, 0, nxt);
            }
            // LDS reads complete in order: with the TM+TN reads of the next set
            // issued last, lgkmcnt(TM+TN) means this set has landed.  (At the
            // last k-step of the last stage nothing newer is pending.)
            ready(f[ks & 1], ks < BK / 16 - 1 || kt + 1 < nk);
            mma(f[ks & 1], KS);
        });
    }
    if constexpr (CHAINS == 4)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][0][r] = (acc[0][0][r] + chain[1][r]) + (chain[2][r] + chain[3][r]);

    const int64_t c_off = (int64_t)batch * p.sC;
    float* ws = p.splits > 1 ? p.ws + (int64_t)blockIdx.z * p.M * p.N : nullptr;
    constexpr int GT = PER_CU * NW > 8 ? 1 : TM * TN;   // four waves to a SIMD: 128 registers each
    store_tiles<EP, TM, TN, GT>(p, acc, reinterpret_cast<float*>(smem) + wave * 32 * CSTAGE, c_off, ws, lane,
                        [&](int i) { return m0 + wm * WM + i * 32; }, [&](int j) { return n0 + wn * WN + j * 32; });
}

// Tiles whose eight waves form two groups of four, one wave of each per SIMD,
// and work in alternating intervals divided by barriers: while one group
// multiplies, the other reads its next fragments from LDS and issues its share
// of the global -> LDS loads, so neither the LDS reads nor the ~16 clocks that a
// load instruction occupies the address unit stand in front of the matrix
// cores.  (With all waves in step, loads and products took turns: 4096^3 with
// 256 x 256 tiles ran 134 us, its loads alone 97, its products alone 99.)
//
// A stage (64 of K) is NA units of UA rows of A and NB units of 128 rows of B.
// Waves form a 2 x 4 grid in each pair of units (group = grid row); a phase,
// one memory and one matrix interval, multiplies one A unit by one B unit.  Each
// unit of the S-slot ring is refilled in the phase after the one that read it
// (reads are waited for before the barrier that ends their interval, so both
// groups are done with it):
//   NB = 2, NA = 2, S = 2 (256 x 256)      NB = 1
//   phase reads        products refills      phase  reads             products refills
//   0     A0           A0 B0    B0           0      A0                A0 B     B, the last A unit
//   1     B1           A0 B1    A0           q      Aq                Aq B     A(q-1)
//   2     A1           A1 B1    B1           last   Aq, B of kt + 1   Aq B     A(q-1)
//   3     B0 of kt + 1 A1 B0    A1
// Loads complete in issue order and every phase issues a fixed number, so "the
// units read next have landed" is a constant vmcnt at the end of each memory
// interval, and nearly the whole ring is in flight.  Loads past the split's K are
// issued out of the descriptor's range: they write zeros to LDS and move
// nothing, which serves the K tail and keeps the counts the same to the end.
template <bool BF16, bool EP, int NA, int NB, int UA, int S>
__global__ __launch_bounds__(512, 2) void gemm_pingpong_kernel(const GemmArgs p) {
    constexpr int BM = NA * UA, BN = NB * 128, BK = 64;
    constexpr int ABYTES = UA * BK * 2, BBYTES = 128 * BK * 2, STAGE = NA * ABYTES + NB * BBYTES;
    constexpr int LA = UA / 64;                        // load instructions per wave of an A unit (2 of a B unit)
    constexpr int TA = UA / 64;                        // 32-row tiles per wave of an A unit (1 column tile of a B unit)
    static_assert((NB == 2 && NA == 2 && S == 2) || (NB == 1 && UA == 64), "phase tables above");
    using G = StageGeom<BK>;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[S * STAGE];
    static_assert(S * STAGE >= 8 * 32 * CSTAGE * 4, "ring too small for the store staging");

    // tile order as in gemm_mfma_kernel
    const int tiles = p.tiles_m * p.tiles_n;
    int t = blockIdx.x;
    const int per = tiles / 8;
    if (t < 8 * per) t = (t % 8) * per + t / 8;
    const int tm = t % p.tiles_m, tn = t / p.tiles_m;
    const int m0 = tm * BM, n0 = tn * BN;
    const int batch = blockIdx.z / p.splits, split = blockIdx.z % p.splits;
    const uint16_t* __restrict__ A = p.A + (int64_t)batch * p.sA;
    const uint16_t* __restrict__ B = p.B + (int64_t)batch * p.sB;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    const int nk_all = (p.K + BK - 1) / BK;
    const int kt0 = split * p.split_stages;
    const int nk = min(nk_all - kt0, p.split_stages);

    const i32x4 rsa = raw_rsrc(A + (int64_t)m0 * p.lda, (uint32_t)((int64_t)(p.M - m0) * p.lda * 2));
    const i32x4 rsb = raw_rsrc(B + (int64_t)n0 * p.ldb, (uint32_t)((int64_t)(p.N - n0) * p.ldb * 2));
    // load instruction g = wave + 8 q of a unit fills its rows 8 g .. 8 g + 7
    const int lrow = 8 * wave + lane / 8;
    const int ls = (lane % 8) ^ G::swz(lrow);          // the same for every q
    uint32_t va[NA][LA], vb[NB][2];                    // byte offsets at K column kt0 * BK
#pragma unroll
    for (int u = 0; u < NA; ++u)
#pragma unroll
        for (int q = 0; q < LA; ++q)
            va[u][q] = (uint32_t)(((int64_t)min(UA * u + 64 * q + lrow, p.M - 1 - m0) * p.lda + kt0 * BK + ls * 8) * 2);
#pragma unroll
    for (int u = 0; u < NB; ++u)
#pragma unroll
        for (int q = 0; q < 2; ++q)
            vb[u][q] = (uint32_t)(((int64_t)min(128 * u + 64 * q + lrow, p.N - 1 - n0) * p.ldb + kt0 * BK + ls * 8) * 2);
    // a lane's 16 bytes of stage kt are in range while kt * BK < klim
    const int klim = min(p.K - kt0 * BK, nk * BK) - ls * 8;
    const uint32_t lds0 = lds_offset(smem);
    const uint32_t wave_lds = lds0 + wave * 1024;
    auto refill_a = [&](int u, uint32_t slot, int kt) {
#pragma unroll
        for (int q = 0; q < LA; ++q)
            asm_buffer_load_lds_b128(rsa, kt * BK < klim ? va[u][q] + kt * (BK * 2) : 0xFFFFFF00u,
                                     wave_lds + slot + u * ABYTES + q * 8192);
    };
    auto refill_b = [&](int u, uint32_t slot, int kt) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
            asm_buffer_load_lds_b128(rsb, kt * BK < klim ? vb[u][q] + kt * (BK * 2) : 0xFFFFFF00u,
                                     wave_lds + slot + NA * ABYTES + u * BBYTES + q * 8192);
    };

    f32x16 acc[NA * TA][NB];
#pragma unroll
    for (int i = 0; i < NA * TA; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    // fragments: row lane & 31 of a 32-row tile, 16-byte slot 2 ks + lane / 32
    uint32_t aaddr[4], baddr[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const uint32_t c = (uint32_t)((2 * ks + (lane >> 5)) ^ G::swz(lane & 31)) << 4;
        aaddr[ks] = lds0 + (wm * (UA / 2) + (lane & 31)) * 128 + c;
        baddr[ks] = lds0 + NA * ABYTES + (wn * 32 + (lane & 31)) * 128 + c;
    }
    // fb: the first B unit of even and odd stages, the second B unit
    u32x4 fa[TA][4], fb[NB + 1][4];
    auto read_a = [&](auto U, uint32_t slot) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            fa[0][ks] = asm_lds_read_b128<decltype(U)::value * ABYTES>(aaddr[ks] + slot);
            if constexpr (TA == 2) fa[1][ks] = asm_lds_read_b128<decltype(U)::value * ABYTES + 4096>(aaddr[ks] + slot);
        }
    };
    auto read_b = [&](auto U, uint32_t slot, u32x4 (&f)[4]) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) f[ks] = asm_lds_read_b128<decltype(U)::value * BBYTES>(baddr[ks] + slot);
    };
    auto pin = [&](u32x4 (&f)[4]) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) asm_pin(f[ks]);
    };
    auto pin_a = [&]() {
        pin(fa[0]);
        if constexpr (TA == 2) pin(fa[1]);
    };
    // end of a memory interval: this wave's reads are done, all but the newest
    // PENDING of its loads have landed
    auto mem_end = [&](auto PENDING) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(PENDING)::value) : "memory");
    };
    auto products = [&](auto I, auto J, u32x4 (&f)[4]) {
        constexpr int i = TA * decltype(I)::value, j = decltype(J)::value;
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int x = 0; x < TA; ++x) acc[i + x][j] = mfma32<BF16>(fa[x][ks], f[ks], acc[i + x][j]);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
    };
    constexpr std::integral_constant<int, 0> c0{};
    constexpr std::integral_constant<int, 1> c1{};
    // stage kt in ring slot `cur` (byte offset); `next` is the slot of kt + 1,
    // `prev` that of kt - 1
    auto stage = [&](int kt, uint32_t prev, uint32_t cur, uint32_t next, u32x4 (&b0)[4], u32x4 (&b0_next)[4]) {
        if constexpr (NB == 2) {
            constexpr std::integral_constant<int, 12> pending{};
            read_a(c0, cur);
            refill_b(0, cur, kt + S);
            mem_end(pending);
            pin_a();
            products(c0, c0, b0);
            read_b(c1, cur, fb[2]);
            refill_a(0, cur, kt + S);
            mem_end(pending);
            pin(fb[2]);
            products(c0, c1, fb[2]);
            read_a(c1, cur);
            refill_b(1, cur, kt + S);
            mem_end(pending);
            pin_a();
            products(c1, c1, fb[2]);
            read_b(c0, next, b0_next);
            refill_a(1, cur, kt + S);
            mem_end(pending);
            pin(b0_next);
            products(c1, c0, b0);
        } else {
            constexpr int L = NA + 2;                  // loads per wave and stage
            static_for<NA>([&](auto Q) {
                constexpr int q = decltype(Q)::value;
                read_a(Q, cur);
                if constexpr (q == NA - 1) read_b(c0, next, b0_next);
                if constexpr (q == 0) {
                    refill_b(0, cur, kt + S);
                    refill_a(NA - 1, prev, kt + S - 1);
                } else {
                    refill_a(q - 1, cur, kt + S);
                }
                mem_end(std::integral_constant<int, (S - 1) * L + (q < NA - 2 ? NA : NA - 2)>{});
                pin_a();
                if constexpr (q == NA - 1) pin(b0_next);
                products(Q, c0, b0);
            });
        }
    };

    // the ring's first stages, in the order the phases issue them
    if constexpr (NB == 2) {
        for (int k = 0; k < S; ++k) {
            refill_b(0, k * STAGE, k);
            refill_a(0, k * STAGE, k);
            refill_b(1, k * STAGE, k);
            refill_a(1, k * STAGE, k);
        }
        asm_wait_vmcnt<12>();
    } else {
        for (int k = 0; k < S; ++k) {
            refill_b(0, k * STAGE, k);
            if (k > 0) refill_a(NA - 1, (k - 1) * STAGE, k - 1);
#pragma unroll
            for (int u = 0; u < NA - 1; ++u) refill_a(u, k * STAGE, k);
        }
        asm_wait_vmcnt<(S - 1) * (NA + 2) + NA - 2>();
    }
    __builtin_amdgcn_s_barrier();
    read_b(c0, 0, fb[0]);
    asm_wait_lgkmcnt<0>();
    pin(fb[0]);
    __builtin_amdgcn_s_barrier();                // B0's slot may be refilled
    if (wm == 1) __builtin_amdgcn_s_barrier();   // the second group runs one interval behind
    uint32_t prev = (S - 1) * STAGE, cur = 0, next = STAGE;
    auto advance = [&]() {
        prev = cur;
        cur = next;
        next = next == (S - 1) * STAGE ? 0 : next + STAGE;
    };
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
        stage(kt, prev, cur, next, fb[0], fb[1]);
        advance();
        stage(kt + 1, prev, cur, next, fb[1], fb[0]);
        advance();
    }
    if (kt < nk) stage(kt, prev, cur, next, fb[0], fb[1]);
    if (wm == 0) __builtin_amdgcn_s_barrier();
    asm_wait_vmcnt<0>();                         // the out-of-range loads write LDS too

    const int64_t c_off = (int64_t)batch * p.sC;
    float* ws = p.splits > 1 ? p.ws + (int64_t)blockIdx.z * p.M * p.N : nullptr;
    store_tiles<EP, NA * TA, NB, NA * TA * NB <= 4 ? NA * TA * NB : 2>(p, acc, reinterpret_cast<float*>(smem) + wave * 32 * CSTAGE, c_off, ws, lane,
                             [&](int i) { return m0 + UA * (i / TA) + wm * (UA / 2) + 32 * (i % TA); },
                             [&](int j) { return n0 + 128 * j + wn * 32; });
}

// Sums the split-K partials in split order (deterministic), applies the
// epilogue and stores C: thread = V consecutive output elements of the
// flattened [M][N] (V = 4 reads the partials as 16-byte vectors; it needs
// M*N % 4 == 0 so every split's partial stays 16-byte aligned).
template <int V, bool EP>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const GemmArgs p) {
    const int64_t mn = (int64_t)p.M * p.N;
    const int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
    const int b = blockIdx.y;
    if (i0 >= mn) return;
    const float* ws = p.ws + (int64_t)b * p.splits * mn + i0;
    if constexpr (V == 4) {
        // N % 4 == 0: the four elements share a row, and with vec_c they are
        // one aligned 16-byte (fp32) or 8-byte (16-bit) piece of C; the
        // operands are requested before the first sum
        if (p.vec_c && p.N % 4 == 0) {
            const int row = (int)(i0 / p.N), col = (int)(i0 - (int64_t)row * p.N);
            const int64_t idx = (int64_t)b * p.sC + (int64_t)row * p.ldc + col;
            f32x4 acc = *reinterpret_cast<const f32x4*>(ws);
            u32x4 bias{}, mul{}, res{};
            if (EP && p.vec_ep) {
                if (p.ep.bias) bias = load_operand4(p.ep.bias, col, p.ep.dtype);
                if (p.ep.mul) mul = load_operand4(p.ep.mul, idx, p.ep.dtype);
                if (p.ep.res) res = load_operand4(p.ep.res, idx, p.ep.dtype);
            }
            for (int s = 1; s < p.splits; ++s) acc += *reinterpret_cast<const f32x4*>(ws + s * mn);
            if (EP && p.vec_ep) acc = combine4(p.ep, activate4(p.ep, acc, bias), mul, res);
            if (EP && !p.vec_ep)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = apply_epilogue(p.ep, acc[e], idx + e, col + e);
            store_c4(p, idx - col, col, acc);
            return;
        }
    }
    float v[V];
    if constexpr (V == 4) {
        f32x4 acc = *reinterpret_cast<const f32x4*>(ws);
        for (int s = 1; s < p.splits; ++s) acc += *reinterpret_cast<const f32x4*>(ws + s * mn);
        v[0] = acc[0]; v[1] = acc[1]; v[2] = acc[2]; v[3] = acc[3];
    } else {
        v[0] = 0.0f;
        for (int s = 0; s < p.splits; ++s) v[0] += ws[s * mn];
    }
#pragma unroll
    for (int e = 0; e < V; ++e) {
        const int64_t i = i0 + e;
        const int row = (int)(i / p.N), col = (int)(i - (int64_t)row * p.N);
        const int64_t idx = (int64_t)b * p.sC + (int64_t)row * p.ldc + col;
        store_out(p.C, idx, EP ? apply_epilogue(p.ep, v[e], idx, col) : v[e], p.c_dtype);
    }
}

// ---- launch configuration ----------------------------------------------------

typedef void (*GemmKernel)(const GemmArgs);

struct TileCfg {
    int bm, bn, bk, stages, waves;
    int per_cu;       // resident blocks per CU (LDS ring and registers)
    int eff;          // TFLOP/s of a round that fills every slot, and what the
    float fixed;      // round takes besides its products (us)
    bool buf;         // buffer-addressed direct loads: operands below 4 GiB only
    GemmKernel kernel[2][2];   // [bf16][epilogue at the store]
};

#define MVLM_TILE(BMv, BNv, BKv, Sv, WMv, WNv, PER_CU, EFF, FIXED)                                              \
    TileCfg{BMv, BNv, BKv, Sv, WMv * WNv, PER_CU, EFF, FIXED, false,                                            \
            {{gemm_mfma_kernel<false, false, BMv, BNv, BKv, Sv, WMv, WNv, PER_CU>,                              \
              gemm_mfma_kernel<false, true, BMv, BNv, BKv, Sv, WMv, WNv, PER_CU>},                              \
             {gemm_mfma_kernel<true, false, BMv, BNv, BKv, Sv, WMv, WNv, PER_CU>,                               \
              gemm_mfma_kernel<true, true, BMv, BNv, BKv, Sv, WMv, WNv, PER_CU>}}}
#define MVLM_PINGPONG(NAv, NBv, UAv, Sv, EFF, FIXED)                                                            \
    TileCfg{NAv * UAv, NBv * 128, 64, Sv, 8, 1, EFF, FIXED, true,                                               \
            {{gemm_pingpong_kernel<false, false, NAv, NBv, UAv, Sv>, gemm_pingpong_kernel<false, true, NAv, NBv, UAv, Sv>}, \
             {gemm_pingpong_kernel<true, false, NAv, NBv, UAv, Sv>, gemm_pingpong_kernel<true, true, NAv, NBv, UAv, Sv>}}}
// All but the last are the automatic choices.  What each costs in plan_gemm's
// model was fitted to the times of every tile and K split over 2100 fp16 products
// (M 1 .. 16384, N 16 .. 51200, K 136 .. 14336; the choice is 1.6% from the
// fastest on average, and 12 products are more than 3% from the better of the
// choice before and the one of the tiles before these).  eff is the rate of a round's products with every slot
// busy, fixed what a round takes besides (first loads, last stores).  Without
// the latter, a 128 x 128 tile whose K is cut into splits of a few stages looked
// faster than it is: 121 x 2945 x 2112 15.6 us with six splits, 13.2 with two of
// 64 x 64 tiles; 66 x 5836 x 1024 11.3 against 8.3 us.  Plain fp16 products, the
// tile's time against the best tile with all waves in step: 4096^3 105 us (256 x 256; 134),
// 1536 x 6144 x 2048 44 (256 x 256; 67), 2048 x 4096 x 600 16.6 (256 x 128; 18.0),
// 768 x 6144 x 2048 26.7 (192 x 128; 31.9), 768 x 8192 x 2048 30.2 (192 x 128;
// 33.7), 729 x 3456 x 1152 13.9 (128 x 128; 14.1), 729 x 4304 x 1152 14.2 (128 x
// 128; 15.3), 2048^3 23.5 (128 x 128; 25.7).  A fifth slot for 128 x 128 (160
// KiB) is slower, 13.9 us at 729 x 3456 x 1152.  Products of few tiles stay with
// 64 x 64, two blocks to a CU: 729 x 1152 x 1152 takes 8.8 us with two 128-wide
// stages, 12.8 with 128 x 128; 64-wide stages serve the many-way K splits of
// few-row products.  128 x 128 in step (two 128-wide stages) serves operands
// beyond the buffer descriptors' 4 GiB, 96 x 192 up to 96 rows by many columns
// (64 x 46656 x 3840 79 us, 86 with 64 x 64).
static const TileCfg kTiles[] = {
    MVLM_PINGPONG(2, 2, 128, 2, 1415, 4.9), MVLM_PINGPONG(4, 1, 64, 3, 990, 2.4),
    MVLM_PINGPONG(3, 1, 64, 4, 905, 2.5), MVLM_PINGPONG(2, 1, 64, 4, 785, 2.5),
    MVLM_TILE(64, 64, 64, 4, 2, 2, 2, 380, 1.4), MVLM_TILE(64, 64, 128, 2, 2, 2, 2, 420, 1.1),
    MVLM_TILE(128, 128, 128, 2, 4, 2, 1, 650, 5.7), MVLM_TILE(96, 192, 128, 2, 3, 2, 1, 535, 3.8),
    MVLM_TILE(128, 128, 32, 4, 4, 2, 2, 690, 2.0),
};
constexpr int kAutoTiles = 8;
#undef MVLM_TILE
#undef MVLM_PINGPONG

struct GemmPlan {
    const TileCfg* tile;
    int splits, split_stages;
};

// The tile and K split with the least modelled time: block rounds x (one
// block's share of the tile's full-chip throughput and the round's fixed cost),
// plus, for a split, writing and re-reading the fp32 partials (3.7 TB/s) and a
// second launch, or else the epilogue, which costs a tile of 32 rows more in the
// store pass than it does that launch (186 x 1300 x 832 with bias and residual
// 9.7 us in one launch, 8.9 in three splits; 186 x 1299 x 832 10.5 and 9.6; with
// 1 us for it 1408 x 448 x 1240 took two splits, 14.4 against 13.1).  MVLM_GEMM_TILE=<bm>x<bn>s<stages>w<waves>[k<bk>] forces a compiled tile
// and MVLM_GEMM_SPLITS=<n> a split count (tuning runs; read at every launch).
static GemmPlan plan_gemm(int M, int N, int K, int batch, int num_cus, bool buf_ok, bool ep) {
    GemmPlan best{&kTiles[4], 1, 0};
    double best_t = 1e30;
    const char* force = std::getenv("MVLM_GEMM_TILE");
    const TileCfg* forced = nullptr;
    if (force) {
        int bm = 0, bn = 0, st = 0, w = 0, bk = 64;
        if (std::sscanf(force, "%dx%ds%dw%dk%d", &bm, &bn, &st, &w, &bk) >= 4)
            for (const TileCfg& c : kTiles)
                if (c.bm == bm && c.bn == bn && c.stages == st && c.waves == w && c.bk == bk && (buf_ok || !c.buf))
                    forced = &c;
    }
    const char* fs = std::getenv("MVLM_GEMM_SPLITS");
    const int forced_splits = fs ? std::atoi(fs) : 0;
    // K <= 128 (e.g. attention scores, head_dim 72): a block's time is its load
    // latency and its C store, not its MFMAs, which the model above does not
    // see; 128x128 tiles with 32-wide stages (less K padding, two blocks per
    // CU) measured fastest there (16 x 729x729x72: 19.9 us vs 25.2 us).
    if (!forced && K <= 128 && forced_splits <= 1)
        for (const TileCfg& c : kTiles)
            if (c.bm == 128 && c.bn == 128 && c.bk == 32 && c.per_cu == 2) forced = &c;
    const int n_cand = forced ? 1 : kAutoTiles;
    for (int i = 0; i < n_cand; ++i) {
        const TileCfg& c = forced ? *forced : kTiles[i];
        if (c.buf && !buf_ok) continue;
        const int nk = (K + c.bk - 1) / c.bk;
        for (int splits : {1, 2, 3, 4, 6, 8}) {
            if (forced_splits > 0 && splits != forced_splits) continue;
            if (splits > 1 && nk < 4 * splits) break;                 // keep at least 4 stages per split
            const int ss = (nk + splits - 1) / splits;
            const int used = (nk + ss - 1) / ss;                         // non-empty splits
            if (used != splits) continue;
            const int64_t tiles = (int64_t)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * batch * splits;
            const int64_t slots = (int64_t)num_cus * c.per_cu;
            const int64_t rounds = (tiles + slots - 1) / slots;
            const double block_flops = 2.0 * c.bm * c.bn * (double)ss * c.bk;
            double t = rounds * (block_flops / (c.eff * 1e12 / (double)slots) + c.fixed * 1e-6);
            if (splits > 1) t += (double)M * N * batch * 4.0 * (2.0 * splits + 1.0) / 3.7e12 + 3.4e-6;
            else if (ep) t += 0.3e-6 * std::min(M, 32) / 32;
            if (t < best_t) { best_t = t; best = GemmPlan{&c, splits, ss}; }
        }
    }
    if (best.split_stages == 0) best.split_stages = (K + best.tile->bk - 1) / best.tile->bk;
    return best;
}

// Copies rows of K elements (row r of batch b at src + b*stride + r*ld) into
// dst [batch][rows][Kp], zero-filling columns K..Kp-1.
__global__ __launch_bounds__(256) void gemm_pad_rows_kernel(const uint16_t* __restrict__ src, int64_t ld,
                                                            int64_t stride, int rows, int K, uint16_t* __restrict__ dst,
                                                            int Kp, int64_t total) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t r = i / Kp;
        const int k = (int)(i - r * Kp);
        const int64_t b = r / rows, rr = r - b * rows;
        dst[i] = k < K ? src[b * stride + rr * ld + k] : (uint16_t)0;
    }
}

// Workspace layout: [split partials][padded A][padded B], each 256-byte aligned.
struct GemmWorkspace {
    bool pad_a = false, pad_b = false;
    int kp = 0;                    // K the kernel runs with (zero columns past K)
    GemmPlan plan{};
    size_t split_bytes = 0, a_off = 0, b_off = 0, total = 0;
};

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

static GemmWorkspace gemm_workspace(int batch, int M, int N, int K, int64_t lda, int64_t ldb, int64_t sA,
                                   int64_t sB, int kread_b, int num_cus, bool ep) {
    GemmWorkspace w;
    const int k8 = (int)round_up(K, 8);
    w.pad_a = K % 8 != 0 || lda % 8 != 0 || (batch > 1 && sA % 8 != 0);
    w.pad_b = ldb % 8 != 0 || (batch > 1 && sB % 8 != 0) || kread_b < k8;
    w.kp = (w.pad_a || w.pad_b) ? k8 : K;
    // buffer-addressed tiles need each operand's rows within a 32-bit byte range
    const int64_t lda_k = w.pad_a ? w.kp : lda, ldb_k = w.pad_b ? w.kp : ldb;
    const bool buf_ok = (int64_t)M * lda_k * 2 < ((int64_t)1 << 32) - 256 && (int64_t)N * ldb_k * 2 < ((int64_t)1 << 32) - 256;
    w.plan = plan_gemm(M, N, w.kp, batch, num_cus > 0 ? num_cus : 256, buf_ok, ep);
    w.split_bytes = w.plan.splits > 1 ? align256((size_t)w.plan.splits * batch * M * N * sizeof(float)) : 0;
    w.a_off = w.split_bytes;
    const size_t a_bytes = w.pad_a ? align256((size_t)batch * M * w.kp * 2) : 0;
    w.b_off = w.a_off + a_bytes;
    const size_t b_bytes = w.pad_b ? align256((size_t)batch * N * w.kp * 2) : 0;
    w.total = w.b_off + b_bytes;
    return w;
}

size_t gemm_workspace_bytes(int batch, int M, int N, int K, int64_t lda, int64_t ldb, int64_t sA, int64_t sB,
                            int kread_b, int num_cus, bool ep) {
    return gemm_workspace(batch, M, N, K, lda, ldb, sA, sB, kread_b, num_cus, ep).total;
}

// The part of C (whole tiles, if one fits) whose split partials fit `room` bytes;
// rows == 0 if not even one row of a tile does.  A launch with less workspace than all partials take
// covers C band by band, with the same tile and splits and so the same sums.
struct GemmBand {
    int rows, cols;
};
static GemmBand gemm_band(const GemmPlan& g, int M, int N, size_t room) {
    const int64_t fit = (int64_t)(room / ((size_t)g.splits * sizeof(float)));   // outputs per band
    if (g.splits == 1 || (int64_t)M * N <= fit) return {M, N};
    const int bm = g.tile->bm, bn = g.tile->bn;
    auto even = [](int64_t all, int64_t most, int64_t tile) {   // as few bands, of nearly one size
        const int64_t bands = (all + most - 1) / most;
        return (int)std::min(all, ((all + bands - 1) / bands + tile - 1) / tile * tile);
    };
    int64_t rows = fit / N / bm * bm, cols = N;
    if (rows == 0) {
        rows = std::min(M, bm);
        cols = fit / rows / bn * bn;
        if (cols == 0) {             // less than a tile: rows of one
            cols = std::min(N, bn);
            rows = fit / cols;
            if (rows == 0) return {0, 0};
            return {(int)rows, even(N, cols, bn)};
        }
    }
    return {even(M, rows, bm), even(N, cols, bn)};
}

// The least workspace a launch runs in.  A split count forced from outside is
// refused where it does not fit whole: a tuning run measures what it asked for.
size_t gemm_workspace_least(int M, int N, int K, int64_t lda, int64_t ldb, int kread_b, int num_cus, bool ep) {
    const GemmWorkspace w = gemm_workspace(1, M, N, K, lda, ldb, 0, 0, kread_b, num_cus, ep);
    if (w.plan.splits == 1 || std::getenv("MVLM_GEMM_SPLITS")) return w.total;
    const size_t row = (size_t)std::min(N, w.plan.tile->bn) * w.plan.splits * sizeof(float);
    return w.total - w.split_bytes + std::min(w.split_bytes, align256(row));
}

// Launches kernel `idx` of an op made of `n` kernels (plan profiling times the
// first kernel's start to the last one's stop).
template <typename... KArgs, typename... Args>
static void launch_seq(int idx, int n, void (*kernel)(KArgs...), dim3 grid, dim3 block, hipStream_t s,
                       Args&&... args) {
    if (n == 1) launch_kernel(kernel, grid, block, 0, s, std::forward<Args>(args)...);
    else launch_kernel_part(idx == 0 ? LaunchPart::First : idx == n - 1 ? LaunchPart::Last : LaunchPart::Middle,
                            kernel, grid, block, 0, s, std::forward<Args>(args)...);
}

static unsigned pad_grid(int64_t total) {
    const int64_t b = (total + 255) / 256;
    return (unsigned)(b < 4096 ? b : 4096);
}

hipError_t launch_gemm_mfma(hipStream_t s, const void* A, int ab_dtype, const void* B, void* C, int c_dtype,
                            int batch, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
                            int64_t strideA, int64_t strideB, int64_t strideC, int kread_b, int num_cus,
                            const Epilogue* ep, void* workspace, size_t workspace_bytes) {
    const GemmWorkspace w = gemm_workspace(batch, M, N, K, lda, ldb, strideA, strideB, kread_b, num_cus, ep && ep->any());
    if (w.total > 0 && !workspace) return hipErrorInvalidValue;
    const GemmPlan& g = w.plan;
    const TileCfg& t = *g.tile;
    GemmBand band{M, N};
    size_t split_bytes = w.split_bytes;
    if (workspace_bytes < w.total) {
        const size_t pads = w.total - w.split_bytes;
        if (batch > 1 || workspace_bytes < pads) return hipErrorInvalidValue;
        split_bytes = (workspace_bytes - pads) & ~(size_t)255;
        band = gemm_band(g, M, N, split_bytes);
        if (band.rows == 0) return hipErrorInvalidValue;
    }
    const size_t a_off = split_bytes, b_off = a_off + (w.b_off - w.a_off);
    GemmArgs a{};
    a.A = (const uint16_t*)A; a.B = (const uint16_t*)B; a.C = C; a.c_dtype = c_dtype;
    a.M = M; a.N = N; a.K = w.kp; a.lda = lda; a.ldb = ldb; a.ldc = ldc;
    a.sA = strideA; a.sB = strideB; a.sC = strideC;
    a.kread_b = kread_b;
    if (ep && ep->any()) {
        a.ep = *ep;
        a.ep_on = 1;
    }
    a.splits = g.splits;
    a.split_stages = g.split_stages;
    a.ws = (float*)workspace;
    {
        const int es = c_dtype == MVLM_F32 ? 4 : 2;
        a.vec_c = ((uintptr_t)C % (4 * es) == 0) && (ldc % 4 == 0) && (strideC % 4 == 0);
        a.vec_ws = N % 4 == 0;   // (of a band too: it ends at C's last column or is whole tiles wide)
        const uintptr_t operands = (uintptr_t)a.ep.bias | (uintptr_t)a.ep.mul | (uintptr_t)a.ep.res;
        a.vec_ep = a.ep_on && a.vec_c && N % 4 == 0 && operands % (4 * es) == 0;
    }
    const int bands = ((M + band.rows - 1) / band.rows) * ((N + band.cols - 1) / band.cols);
    const int n = (int)w.pad_a + (int)w.pad_b + bands * (g.splits > 1 ? 2 : 1);
    int idx = 0;
    if (w.pad_a) {
        uint16_t* ap = (uint16_t*)((char*)workspace + a_off);
        const int64_t total = (int64_t)batch * M * w.kp;
        launch_seq(idx++, n, gemm_pad_rows_kernel, dim3(pad_grid(total)), dim3(256), s, (const uint16_t*)A, lda,
                   strideA, M, K, ap, w.kp, total);
        a.A = ap; a.lda = w.kp; a.sA = (int64_t)M * w.kp;
    }
    if (w.pad_b) {
        uint16_t* bp = (uint16_t*)((char*)workspace + b_off);
        const int64_t total = (int64_t)batch * N * w.kp;
        launch_seq(idx++, n, gemm_pad_rows_kernel, dim3(pad_grid(total)), dim3(256), s, (const uint16_t*)B, ldb,
                   strideB, N, min(K, kread_b), bp, w.kp, total);
        a.B = bp; a.ldb = w.kp; a.sB = (int64_t)N * w.kp; a.kread_b = w.kp;
    }
    const GemmKernel k = t.kernel[ab_dtype == MVLM_BF16][a.ep_on && g.splits == 1];
    const size_t cs = dtype_size(c_dtype);
    auto at = [](const void* base, int64_t offset) { return base ? (const char*)base + offset : nullptr; };
    for (int r0 = 0; r0 < M; r0 += band.rows)
        for (int c0 = 0; c0 < N; c0 += band.cols) {
            GemmArgs b = a;
            const int64_t c_off = ((int64_t)r0 * ldc + c0) * (int64_t)cs;
            b.M = std::min(band.rows, M - r0);
            b.N = std::min(band.cols, N - c0);
            b.A = a.A + (int64_t)r0 * a.lda;
            b.B = a.B + (int64_t)c0 * a.ldb;
            b.C = (char*)C + c_off;
            b.ep.bias = at(a.ep.bias, c0 * (int64_t)cs);
            b.ep.mul = at(a.ep.mul, c_off);
            b.ep.res = at(a.ep.res, c_off);
            b.tiles_m = (b.M + t.bm - 1) / t.bm;
            b.tiles_n = (b.N + t.bn - 1) / t.bn;
            launch_seq(idx++, n, k, dim3((unsigned)(b.tiles_m * b.tiles_n), 1, (unsigned)(batch * g.splits)),
                       dim3(64 * t.waves), s, b);
            if (g.splits > 1) {
                const int64_t mn = (int64_t)b.M * b.N;
                const int v = mn % 4 == 0 ? 4 : 1;
                const auto reduce = v == 4 ? (a.ep_on ? gemm_splitk_reduce_kernel<4, true> : gemm_splitk_reduce_kernel<4, false>)
                                           : (a.ep_on ? gemm_splitk_reduce_kernel<1, true> : gemm_splitk_reduce_kernel<1, false>);
                launch_seq(idx++, n, reduce, dim3((unsigned)((mn / v + 255) / 256), (unsigned)batch), dim3(256), s, b);
            }
        }
    return hipGetLastError();
}

}  // namespace mvlm
