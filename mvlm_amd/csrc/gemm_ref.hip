// The reference's exact-arithmetic GEMM entry points on gfx950.
//
// gemm_naive (src/kernels/gemm.cl:26-51) and gemm_tiled (gemm.cl:74-136)
// compute, per output, acc = fma(A[row,k], B[k,col], acc) over k = 0..K-1 in
// fp32 from fp16 inputs and store RNE fp16.  gemm_order_kernel keeps that exact
// per-output fma sequence, so its results are bit-identical to a CPU
// restatement; only the work partition differs.
//   A [M,K], B [K,N], C [M,N], fp16 row-major.
// gemv_exact keeps the reference gemv's split of K over 256 partial sums and
// its fold order on the packed fp16 weight.
#include "common.h"
#include "device_math.h"

#include <algorithm>

namespace mvlm {

// The products run on v_mfma_f32_16x16x4_f32.  The product of two widened
// fp16 values is exact in fp32, and that instruction adds its four products to
// the accumulator one after another in ascending k, each sum rounded to
// nearest even (checked bit by bit against the fma chain over random, wide
// range, subnormal and infinite inputs), so a chain of them is the reference's
// fma sequence at twice the vector ALU's fp32 rate (256 flops per CU and
// clock).  Zeros past K leave an accumulator as it is: it is never -0, since
// it starts at +0 and a sum of two values of opposite sign that cancels is +0.
//
// Bound: the fp32 matrix rate (157 TFLOP/s at 2.4 GHz).  An MFMA occupies its
// SIMD for 32 cycles, which leaves room for the two 2-byte LDS reads and the
// two conversions that feed it, so operands stay fp16 in LDS in the layout
// they have in memory and are widened on the way into registers.  A block of
// NW waves owns a BM x BN tile of C, a wave TM x TN tiles of 16 x 16; the next
// BK-wide slice of A and B is in flight to registers while the current one is
// multiplied, and the LDS slices alternate (one barrier per slice).  2048^3:
// 399 -> 154 us (43 -> 112 TFLOP/s) against the vector-ALU kernel of 64 x 64
// tiles this replaces; 256^3 36 -> 5.2 us, 32 x 2048 x 2048 253 -> 22 us,
// rows off the 16-byte grid (1500^3) 293 -> 101 us.
// Operand layout: lane l supplies A[l%16][k + l/16] and B[k + l/16][l%16];
// accumulator register i of lane l is C[4*(l/16) + i][l%16].
// Rows start at any 2-byte address (or odd byte, in a view): 16-byte loads take
// unaligned addresses here, and only the chunk at the end of a row is read
// element by element.
template <int BM, int BN, int BK, int WGM, int WGN>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_order_kernel(const uint16_t* __restrict__ A,
                                                                    const uint16_t* __restrict__ B,
                                                                    uint16_t* __restrict__ C, int M, int N, int K,
                                                                    int tiles_m) {
    constexpr int NT = 64 * WGM * WGN;
    constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
    // LDS pitches (elements): the 16 rows x 4 k of an A read and the 4 k x 16
    // columns of a B read fall on distinct banks
    constexpr int PA = BK + 4, PB = BN + 16;
    constexpr int CA = BM * BK / 8 / NT, CB = BK * BN / 8 / NT;   // 8-element chunks per thread and slice
    static_assert(CA >= 1 && CB >= 1 && CA * 8 * NT == BM * BK && CB * 8 * NT == BK * BN, "chunks per thread");
    __shared__ __attribute__((aligned(16))) uint16_t As[2][BM * PA];
    __shared__ __attribute__((aligned(16))) uint16_t Bs[2][BK * PB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, q = lane >> 4;
    const int wm = (wave / WGN) * WM, wn = (wave % WGN) * WN;
    // each XCD takes a contiguous run of tiles, the M tiles of one column of
    // tiles next to each other (they read the same columns of B)
    int t = blockIdx.x;
    const int per = (int)gridDim.x / 8;
    if (t < 8 * per) t = (t % 8) * per + t / 8;
    const int m0 = (t % tiles_m) * BM, n0 = (t / tiles_m) * BN;

    u32x4 ra[CA], rb[CB];
    auto load8 = [](const uint16_t* p, int left) {   // p[0..8), zeros from `left` on
        u32x4 v = {0u, 0u, 0u, 0u};
        if (left >= 8) {
            __builtin_memcpy(&v, p, 16);
        } else if (left > 0) {
#pragma unroll
            for (int e = 0; e < 7; ++e)
                if (e < left) v[e >> 1] |= (uint32_t)p[e] << (16 * (e & 1));
        }
        return v;
    };
    auto load = [&](int k0) {                         // k0 < K: sums with it stay off int's end
#pragma unroll
        for (int c = 0; c < CA; ++c) {
            const int i = tid + c * NT, r = i / (BK / 8), k = 8 * (i % (BK / 8));
            ra[c] = load8(A + (int64_t)(m0 + r) * K + k0 + k, m0 + r < M ? K - k0 - k : 0);
        }
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            const int i = tid + c * NT, k = i / (BN / 8), n = n0 + 8 * (i % (BN / 8));
            rb[c] = load8(B + ((int64_t)k0 + k) * N + n, k < K - k0 ? N - n : 0);
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int c = 0; c < CA; ++c) {
            const int i = tid + c * NT;
            uint16_t* d = As[buf] + (i / (BK / 8)) * PA + 8 * (i % (BK / 8));   // 8-byte aligned
            *reinterpret_cast<u32x2*>(d) = u32x2{ra[c][0], ra[c][1]};
            *reinterpret_cast<u32x2*>(d + 4) = u32x2{ra[c][2], ra[c][3]};
        }
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            const int i = tid + c * NT;
            *reinterpret_cast<u32x4*>(Bs[buf] + (i / (BN / 8)) * PB + 8 * (i % (BN / 8))) = rb[c];
        }
    };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    load(0);
    store(0);
    __syncthreads();
    uint32_t buf = 0;
    for (uint32_t k0 = 0; k0 < (uint32_t)K; k0 += BK, buf ^= 1) {   // (an int would overflow past the last slice)
        const bool more = k0 + BK < (uint32_t)K;
        if (more) load((int)(k0 + BK));
        const uint16_t* as = As[buf] + (wm + l16) * PA + q;
        const uint16_t* bs = Bs[buf] + q * PB + wn + l16;
#pragma unroll
        for (int k = 0; k < BK; k += 4) {
            float a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = f16_bits_to_f32(as[16 * i * PA + k]);
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = f16_bits_to_f32(bs[k * PB + 16 * j]);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        // the other slice was last read before the barrier that ended the
        // previous round
        if (more) store(buf ^ 1);
        __syncthreads();
    }
    constexpr int PC = WN + 8;                        // pitch of a wave's 16 rows of C
    static_assert(NT / 64 * 16 * PC <= 2 * BM * PA || NT / 64 * 16 * PC <= 2 * BK * PB, "staging");
    // Through LDS, 16 rows of the wave at a time, stored as 16-byte pieces (two
    // bytes at a time from the accumulators 2048 x 2048 x 8 took 9.2 us, now 6.5);
    // the loop's last barrier ended the reads of the slices.  A region of its own
    // per wave needs no further barrier: through one tile of the whole block
    // 2048^3 took 161 us, so 154.
    uint16_t* const cw = (NT / 64 * 16 * PC <= 2 * BM * PA ? As[0] : Bs[0]) + wave * 16 * PC;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) cw[(4 * q + r) * PC + 16 * j + l16] = f32_to_f16_bits(acc[i][j][r]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave's writes, before its reads
#pragma unroll
        for (int c = lane; c < 16 * WN / 8; c += 64) {
            const int row = m0 + wm + 16 * i + c / (WN / 8), col = n0 + wn + 8 * (c % (WN / 8));
            if (row >= M || col >= N) continue;
            const uint16_t* v = cw + (c / (WN / 8)) * PC + 8 * (c % (WN / 8));
            uint16_t* out = C + (int64_t)row * N + col;
            if (N - col >= 8) {
                u32x4 t = *reinterpret_cast<const u32x4*>(v);
                __builtin_memcpy(out, &t, 16);
            } else {
                for (int e = 0; e < N - col; ++e) out[e] = v[e];
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // its reads, before the next rows' writes
    }
}

template <int BM, int BN, int BK, int WGM, int WGN>
static hipError_t launch_order(hipStream_t s, const uint16_t* A, const uint16_t* B, uint16_t* C, int M, int N, int K) {
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    launch_kernel(gemm_order_kernel<BM, BN, BK, WGM, WGN>, dim3((unsigned)(tiles_m * tiles_n)), dim3(64 * WGM * WGN), 0, s,
                  A, B, C, M, N, K, tiles_m);
    return hipGetLastError();
}

// Serves mvlm_gemm_naive and mvlm_gemm_tiled.  The tile with the least work on
// the busiest CU: its blocks times what a block takes, the smaller tiles weighted
// by the operand bytes they move per product, plus a block's fixed time and no
// less than one slice of K (4096 x 4096: 17.0, 27.1 and 57.5 us with tiles of 128,
// 64 and 32 at K = 32).  1024^3 takes 256 blocks of 64 (30 us), 2048^3 256 of 128,
// 1500 x 1500 x 8 144 of 128 (6.7 us; 10.2 with 2209 of 32, which the products
// alone would take).
hipError_t launch_gemm_order(hipStream_t s, const uint16_t* A, const uint16_t* B, uint16_t* C, int M, int N, int K,
                             int num_cus) {
    const int cus = num_cus > 0 ? num_cus : 256;
    auto cost = [&](int edge, int bk, double fixed, double slice) {   // us a block, us a slice
        const int64_t tiles = (int64_t)((M + edge - 1) / edge) * ((N + edge - 1) / edge);
        return (double)((tiles + cus - 1) / cus) * (fixed + slice * std::max(1.0, (double)K / bk));
    };
    const double c128 = cost(128, 32, 1.18, 2.09), c64 = cost(64, 64, 0.31, 1.15), c32 = cost(32, 128, 0.08, 0.705);
    if (c128 <= c64 && c128 <= c32) return launch_order<128, 128, 32, 4, 2>(s, A, B, C, M, N, K);
    if (c64 <= c32) return launch_order<64, 64, 64, 2, 2>(s, A, B, C, M, N, K);
    return launch_order<32, 32, 128, 2, 2>(s, A, B, C, M, N, K);
}

// gemv (gemm.cl:215-270) as launched by dispatch_gemv (compute.cpp:141-147):
// y[n] = sum_k x[k] W[n,k] with the reference's summation order.  There, one
// 256-item group owns 4 outputs; item L keeps p = fma(x[k], W[n,k], p) over
// k = L, L+256, L+512, ... and the 256 partials are then folded by
// red[L] = red[L] + red[L+s] for s = 128, 64, ..., 1.
//
// Here one wave owns GX_ROWS outputs of the packed [N][ld] fp16 weight (rows
// zero padded to ld = K rounded up to 64, 128-byte aligned) and streams
// them: lane l holds the partials L = 4l + c, c = 0..3, and in the window
// starting at k0 reads W[n, k0+4l .. k0+4l+3] and the same x quad, one 8-byte
// load each, so a wave's loads are 512 contiguous bytes per row and every
// partial sees the reference's fma sequence.  GX_WIN windows are loaded
// before any is used.  The fold keeps the reference's pairs: strides 128..4
// pair lane l with lane l + s/4 (lane shuffles), strides 2 and 1 pair the
// four partials of lane 0.  Those pairs fix every rounding, so y is
// bit-identical to the reference's.
constexpr int GX_ROWS = 2;   // outputs per wave
constexpr int GX_WIN = 8;    // 256-wide k windows loaded together

template <int WIN>
__device__ __forceinline__ void gemv_exact_windows(const uint16_t* __restrict__ x, const uint16_t* const* rows,
                                                   int k0, int lane, float (&p)[GX_ROWS][4]) {
    uint2 w[WIN][GX_ROWS], xq[WIN];
#pragma unroll
    for (int v = 0; v < WIN; ++v) {
        const int k = k0 + 256 * v + 4 * lane;
        xq[v] = *reinterpret_cast<const uint2*>(x + k);
#pragma unroll
        for (int r = 0; r < GX_ROWS; ++r) w[v][r] = *reinterpret_cast<const uint2*>(rows[r] + k);
    }
    __builtin_amdgcn_sched_barrier(0);   // every load of the windows is issued before the first use
#pragma unroll
    for (int v = 0; v < WIN; ++v) {
        const float xf[4] = {f16_bits_to_f32(xq[v].x & 0xFFFF), f16_bits_to_f32(xq[v].x >> 16),
                             f16_bits_to_f32(xq[v].y & 0xFFFF), f16_bits_to_f32(xq[v].y >> 16)};
#pragma unroll
        for (int r = 0; r < GX_ROWS; ++r) {
            const float wf[4] = {f16_bits_to_f32(w[v][r].x & 0xFFFF), f16_bits_to_f32(w[v][r].x >> 16),
                                 f16_bits_to_f32(w[v][r].y & 0xFFFF), f16_bits_to_f32(w[v][r].y >> 16)};
#pragma unroll
            for (int c = 0; c < 4; ++c) p[r][c] = __builtin_fmaf(xf[c], wf[c], p[r][c]);
        }
    }
}

__global__ __launch_bounds__(256) void gemv_exact_kernel(const uint16_t* __restrict__ x,
                                                         const uint16_t* __restrict__ W, int64_t ld,
                                                         uint16_t* __restrict__ y, int N, int K) {
    const int lane = threadIdx.x & 63;
    const int n0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * GX_ROWS;
    if (n0 >= N) return;   // no block-wide barrier follows
    const uint16_t* rows[GX_ROWS];
#pragma unroll
    for (int r = 0; r < GX_ROWS; ++r) rows[r] = W + (int64_t)min(n0 + r, N - 1) * ld;
    float p[GX_ROWS][4];
#pragma unroll
    for (int r = 0; r < GX_ROWS; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) p[r][c] = 0.0f;
    int k0 = 0;
    for (; k0 + 256 * GX_WIN <= K; k0 += 256 * GX_WIN) gemv_exact_windows<GX_WIN>(x, rows, k0, lane, p);
    for (; k0 + 256 <= K; k0 += 256) gemv_exact_windows<1>(x, rows, k0, lane, p);
    if (k0 < K) {   // the last, partial window: element loads below K only
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int k = k0 + 4 * lane + c;
            if (k < K) {
                const float xv = f16_bits_to_f32(x[k]);
#pragma unroll
                for (int r = 0; r < GX_ROWS; ++r)
                    p[r][c] = __builtin_fmaf(xv, f16_bits_to_f32(rows[r][k]), p[r][c]);
            }
        }
    }
    // lane l < d receives the partial of lane l + d: d = 32 .. 1 are the strides 128 .. 4
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
#pragma unroll
        for (int r = 0; r < GX_ROWS; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) p[r][c] = p[r][c] + __shfl_down(p[r][c], d, 64);
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < GX_ROWS; ++r)
            if (n0 + r < N) y[n0 + r] = f32_to_f16_bits((p[r][0] + p[r][2]) + (p[r][1] + p[r][3]));
    }
}

hipError_t launch_gemv_exact(hipStream_t s, const uint16_t* x, const mvlm_weight* W, uint16_t* y) {
    const int per_block = 4 * GX_ROWS;
    dim3 grid((W->N + per_block - 1) / per_block);
    launch_kernel(gemv_exact_kernel, grid, dim3(256), 0, s, x, (const uint16_t*)W->data, (int64_t)W->ld, y,
                  W->N, W->K);
    return hipGetLastError();
}

}  // namespace mvlm
