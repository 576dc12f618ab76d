// Dequantizing skinny GEMM over GGUF Q8_0 / Q4_0 weights on the matrix cores:
// Y[m][n] = sum_k X[m][k] * w(n, k), 1 <= M <= 16, X and Y fp32 row-major.
//
// The reference plans this kernel (README.md:57, PLAN.md:65) but never wrote
// it.  With M > 1 the fp32 vector ALU would spend 2*M flops per streamed
// weight (M = 16: 42 GFLOP per Phi-1.5 step, ~270 us at the fp32 peak), so
// the products go to v_mfma_f32_16x16x32_bf16 instead, with no loss of
// precision:
//  * codes are small integers (Q8_0: -127..127, Q4_0: c - 8 in -8..7), exact
//    in bf16;
//  * x is split into three bf16 parts x = x1 + x2 + x3 (each the top 16 bits
//    of the remaining fp32 residual; the residuals are exact), which carries
//    24 significant bits, fp32's own precision, over fp32's exponent range;
//  * bf16 x bf16 products are exact in fp32 and the MFMA accumulates in fp32;
//  * the block scale d (fp16, exact in fp32) is applied once per block of 32
//    weights: acc += d * (sum over the block), as in the M = 1 kernel;
//  * Q4_0 multiplies the raw nibbles c and subtracts 8 * (sum of x over the
//    block), that sum coming from one more product of the split x with a
//    ones operand.
// One MFMA covers 16 weight rows x one block of 32 weights x 16 rows of X.
//
// Two kernels share that arithmetic, chosen per launch by size (skinny_keeps_x).
// The one in gemm_skinny_kwalk.hip reads X again for every one to four row groups
// of the weight; the one here keeps X in registers.  Their sums over a block are
// the same, the order of the blocks is not: the last bits of an output depend on
// the kernel and so on what else its launch holds, its error (2-norm against 64
// bits, 1.0e-7 to 1.2e-7 for Q8_0, 1.4e-7 to 1.8e-7 for Q4_0 over K = 512 ..
// 14336) does not.
//
// Operand layout of v_mfma_f32_16x16x32_bf16: lane l supplies
// A[l%16][8*(l/16) .. +7] and B[8*(l/16) .. +7][l%16]; accumulator register i
// of lane l is D[4*(l/16) + i][l%16].  Here A = X (row m = l%16) and B = w^T
// (weight row n0 + l%16).  The k order inside a block is free as long as both
// operands share it: Q8_0 lanes take bytes 8q..8q+7 of the block (q = l/16);
// Q4_0 lanes take its bytes 4q..4q+3, i.e. weights 4q..4q+3 (low nibbles) and
// 16+4q..16+4q+3 (high nibbles).
//
// A workgroup of 8 waves spans up to 64 blocks of K (a chunk of 2048 weights;
// longer rows are cut into equal chunks), eight blocks a wave: the wave loads and
// splits its 16 x 256 slice of X once (96 registers) and then streams the same
// columns of one 16-row group of the weight after another.  Reading X again for
// every row group, as the other kernel does, costs 4 * M * K bytes per row group,
// 14 times the Q4_0 codes of the group at M = 16, and that traffic (from L2,
// through the CU's one vector cache) sets the time of a launch of many row
// groups.  The waves' partial tiles meet in LDS after every four row groups.  One
// workgroup per CU; the row groups of a launch are dealt out in whole rounds (up
// to 14 row groups per workgroup).
//
// Against the other kernel alone, a Phi-1.5 step (49 grouped launches) of M = 16
// went 831 -> 650 us (Q4_0) and 867 -> 701 us (Q8_0), of M = 8 785 -> 592 and 806
// -> 648 us, its LM head 39 -> 22 and 39 -> 27 us.  What bounds a launch now (time
// stamps of the M = 16 QKV + fc1 launch, 10.5 us): 128 KiB of X into every CU and
// its split, 5 us before the first products, then 0.8 us (Q4_0, vector ALU and
// matrix core in turn) to 1.2 us (Q8_0, HBM) per row group.  Sixteen waves of
// four blocks each spend longer in the barriers (Q4_0 M = 16 707 us, Q8_0 691
// us); codes requested before X, with deeper rings, delay X by more than they
// gain (697 and 822 us).  A wave loads eight blocks of X and codes even where it
// owns fewer (rows below 2048 weights), which costs little of that, but makes up
// most of a launch of short rows: the other kernel's part.
//
// Codes go to the wave's own LDS ring with direct 16-byte loads, several row
// groups ahead, and are read back per lane (loading the MFMA layout straight
// from HBM, 16 rows x 32 bytes per instruction, ran at ~1 TB/s whatever the
// arithmetic).  The workgroup's scales are staged once.
//
// Rows of more than one chunk (K > 2048): a workgroup takes one chunk of its
// rows and writes its sums to the device workspace, and a second launch adds
// the chunks in order and applies the epilogue.  Without workspace the launch
// goes to the other kernel.
#include "gemm_skinny.h"

#include <algorithm>
#include <cstdlib>

namespace mvlm {

// Barrier that orders the workgroup's LDS accesses and leaves loads from
// memory in flight (__syncthreads() would wait for all of them).
__device__ __forceinline__ void block_sync() {
    asm_wait_lgkmcnt<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

constexpr int SK_WAVES = 8;                           // waves of a workgroup
constexpr int SK_KB = 8;                              // blocks of K per wave, at most
constexpr int SK_CHUNK = SK_WAVES * SK_KB;            // blocks of K per chunk, at most
constexpr int SK_MAX_RG = 14;                         // row groups per workgroup, at most
constexpr int SK_BATCH = 4;                           // row groups whose partial tiles meet at one barrier
// a row's staged scales of one chunk: 64 fp16 and one more where the chunk
// starts at an odd block, in dwords
constexpr int SK_SCALE_DW = SK_CHUNK / 2 + 2;
constexpr int SK_SCALE_ROWS = 16 * SK_SCALE_DW * 4;   // bytes of a row group's
constexpr int SK_PART_BYTES = SK_BATCH * SK_WAVES * 1024;
constexpr int SK_EP_LOADS = 5;                        // epilogue operands of a thread's two outputs
constexpr int SK_EP_BYTES = SK_EP_LOADS * SK_WAVES * 256;

template <bool Q4>
struct SkinnyLayout {
    static constexpr int BB = Q4 ? 16 : 32;           // code bytes per block per row
    static constexpr int CB = SK_KB * BB;             // code bytes per row per wave (128 / 256)
    static constexpr int P = CB / 16;                 // 16-byte pieces per row
    static constexpr int RPI = 64 / P;                // rows per direct-load instruction
    static constexpr int NDMA = 16 / RPI;             // direct loads per row group
    static constexpr int SLOT = 16 * CB;              // bytes of one row group's codes
    static constexpr int DEPTH = Q4 ? 4 : 2;          // row groups in flight: 64 KiB per CU
    static constexpr int LDS = SK_PART_BYTES + SK_EP_BYTES + SK_MAX_RG * SK_SCALE_ROWS + SK_WAVES * DEPTH * SLOT;
    // Physical piece of logical piece p in LDS row r: XOR-swizzled with row
    // bits so the rows of a read land on distinct banks.
    __device__ static int piece(int p, int r) { return p ^ (Q4 ? (r >> 1) & 7 : r & 15); }
};
static_assert(SkinnyLayout<true>::LDS <= 160 * 1024 && SkinnyLayout<false>::LDS <= 160 * 1024, "LDS of a CU");

// One problem of a (possibly grouped) launch: Y[M][N] = X[M][K] w^T.
struct SkinnyProblem {
    const float* X;
    const uint8_t* codes;
    const uint16_t* scales;
    float* Y;
    float* part;                   // [chunks][M][N] sums of the chunks; null if there is one
    uint32_t ld;                   // code bytes per row
    int N, nb;                     // rows, blocks of K
    int chunks, chunk_blocks;      // chunks of K and blocks per chunk (the last may have fewer)
    uint32_t chunk_div;            // ceil(2^32 / chunks): b / chunks = b * chunk_div >> 32
    int rows;                      // row groups per workgroup
    int ep_on;
    Epilogue ep;
};
struct SkinnyGroup {
    int count, M;
    int block_begin[SKINNY_MAX_GROUP];   // first workgroup of each problem in the grid
    SkinnyProblem p[SKINNY_MAX_GROUP];
};

template <bool Q4>
__global__ __launch_bounds__(64 * SK_WAVES) void gemm_skinny_kernel(const SkinnyGroup g) {
    using L = SkinnyLayout<Q4>;
    extern __shared__ __attribute__((aligned(256))) uint8_t lds[];
    float* const part = reinterpret_cast<float*>(lds);

    int pi = 0;                                       // workgroups are dealt to the problems in order
#pragma unroll
    for (int i = 1; i < SKINNY_MAX_GROUP; ++i)
        if (i < g.count && (int)blockIdx.x >= g.block_begin[i]) pi = i;
    const SkinnyProblem& P = g.p[pi];
    const int M = g.M, N = P.N, nb = P.nb, chunks = P.chunks, chunk_blocks = P.chunk_blocks, rows = P.rows;
    const uint32_t ld = P.ld, chunk_div = P.chunk_div;
    float* const cpart = P.part;
    const float* const X = P.X;
    const uint8_t* const codes = P.codes;
    const uint16_t* const scales = P.scales;
    const bool ep_on = P.ep_on && !cpart;
    // one round trip for the fields, before anything waits for one of them
    asm volatile("" ::"s"(N), "s"(nb), "s"(chunks), "s"(chunk_blocks), "s"(rows), "s"(ld), "s"(chunk_div), "s"(cpart),
                 "s"(X), "s"(codes), "s"(scales));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, q = lane >> 4;

    // this workgroup's row groups [rg0, rg0 + units) and chunk c
    const int bid = (int)blockIdx.x - g.block_begin[pi];
    const int range = chunks > 1 ? (int)__umulhi((uint32_t)bid, chunk_div) : bid;
    const int c = bid - range * chunks;
    const int rg0 = range * rows;
    const int units = min(rows, (N + 15) / 16 - rg0);
    const int n0 = 16 * rg0;

    // Codes, scales and X are read through buffer descriptors (32-bit offsets;
    // the host keeps all three below 2 GiB).
    const i32x4 crs = raw_rsrc(codes, (uint32_t)N * ld);
    const i32x4 srs = raw_rsrc(scales, ((uint32_t)N * (uint32_t)nb * 2 + 3) & ~3u);   // the allocation is padded
    const i32x4 xrs = raw_rsrc(X, (uint32_t)M * (uint32_t)nb * 128);
    const uint32_t ep_base = lds_offset(lds) + SK_PART_BYTES + (uint32_t)(wave * SK_EP_LOADS * 256);
    const uint32_t scale_base = lds_offset(lds) + SK_PART_BYTES + SK_EP_BYTES;
    const uint32_t ring = scale_base + SK_MAX_RG * SK_SCALE_ROWS + (uint32_t)(wave * L::DEPTH * L::SLOT);
    // lanes whose X row is past M read row M - 1: they only feed output rows
    // m >= M, which are never stored
    const int xm = min(l16, M - 1);
    // Lanes of odd rows load their two X pieces in swapped order, so the 16
    // lanes of a quarter-wave (16 rows, one q) read two different offsets of
    // their lines instead of one (the vector cache serves many lines at one
    // offset one after another).
    const bool xodd = (xm & 1) != 0;
    const int x0 = Q4 ? 4 * q : 8 * q, x1 = Q4 ? 16 + 4 * q : 8 * q + 4;
    const int dma_row = lane / L::P, dma_piece = lane % L::P;

    // The waves sum the partial tiles of a batch of row groups and store them:
    // waves 2 k and 2 k + 1 those of row group k of the batch, a lane the
    // outputs (om, l16) and (om + 4, l16).  Their epilogue operands come in by
    // direct 4-byte loads, a batch ahead (absent ones repeat a scale).
    const int om = 8 * (wave & 1) + q, duty = wave >> 1;
    const bool ep = ep_on && 8 * (wave & 1) < M;
    auto issue_ep = [&](int u) {
        const int n = min(n0 + 16 * u + l16, N - 1);
        const float* none = reinterpret_cast<const float*>(scales);
        const int64_t i0 = (int64_t)min(om, M - 1) * N + n, i1 = (int64_t)min(om + 4, M - 1) * N + n;
        const float *b = (const float*)P.ep.bias, *m = (const float*)P.ep.mul, *r = (const float*)P.ep.res;
        const uint32_t dst = __builtin_amdgcn_readfirstlane(ep_base);
        asm_global_load_lds_b32(b ? b + n : none, dst);
        asm_global_load_lds_b32(m ? m + i0 : none, dst + 256);
        asm_global_load_lds_b32(m ? m + i1 : none, dst + 512);
        asm_global_load_lds_b32(r ? r + i0 : none, dst + 768);
        asm_global_load_lds_b32(r ? r + i1 : none, dst + 1024);
    };

    u32x4 xp[SK_KB][3];                               // the wave's slice of X in three bf16 parts
    f32x4 sx[SK_KB];                                  // Q4_0: -8 times its block sums
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};

    const int cb0 = c * chunk_blocks, cb = min(chunk_blocks, nb - cb0);
    const int per = (cb + SK_WAVES - 1) / SK_WAVES;
    const int cnt = max(0, min(per, cb - wave * per));   // this wave's blocks
    const int b0 = cb0 + wave * per;

    // a lane's byte of the codes for each direct load of row group 0,
    // and its last one in bounds (rows past N repeat row N - 1)
    uint32_t voff[L::NDMA], vmax[L::NDMA];
#pragma unroll
    for (int t = 0; t < L::NDMA; ++t) {
        const int r = t * L::RPI + dma_row;
        const uint32_t off = (uint32_t)min(b0 * L::BB + 16 * L::piece(dma_piece, r), nb * L::BB - 16);
        voff[t] = (uint32_t)(n0 + r) * ld + off;
        vmax[t] = (uint32_t)(N - 1) * ld + off;
    }
    auto issue = [&](int u, int slot) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane(ring + (uint32_t)(slot * L::SLOT));
#pragma unroll
        for (int t = 0; t < L::NDMA; ++t)
            asm_buffer_load_lds_b128(crs, min(voff[t] + (uint32_t)(16 * u) * ld, vmax[t]), dst + t * 1024);
    };

    // The scales, the first epilogue operands, X, then the first row
    // groups of codes (past the last one, and in waves without blocks,
    // the clamped addresses repeat loads: no branch may stand between
    // the X loads and the wait for them, where the compiler could move
    // their registers).  Scales: dwords of the rows' scales of this
    // chunk, from the dword its first block lies in; past the array
    // they are clamped to its last dword.
    {
        const int total = units * 16 * SK_SCALE_DW;
        const uint32_t last = ((uint32_t)N * (uint32_t)nb * 2 - 1) & ~3u;
        for (int i = wave * 64; i < total; i += 64 * SK_WAVES) {
            const uint32_t e = (uint32_t)min(i + lane, total - 1), r = e / SK_SCALE_DW, dw = e - r * SK_SCALE_DW;
            const uint32_t row = min((uint32_t)n0 + r, (uint32_t)(N - 1));
            const uint32_t off = (((row * (uint32_t)nb + (uint32_t)cb0) * 2) & ~3u) + 4 * dw;
            asm_buffer_load_lds_b32(srs, min(off, last),
                                    __builtin_amdgcn_readfirstlane(scale_base + 4u * (uint32_t)i));
        }
    }
    if (ep && duty < units) issue_ep(duty);
    u32x4 xr[SK_KB][2];
#pragma unroll
    for (int j = 0; j < SK_KB; ++j) {
        const uint32_t base = (uint32_t)(xm * nb + min(b0 + j, nb - 1)) * 128u;
        xr[j][0] = asm_buffer_load_b128(xrs, base + 4u * (uint32_t)(xodd ? x1 : x0));
        xr[j][1] = asm_buffer_load_b128(xrs, base + 4u * (uint32_t)(xodd ? x0 : x1));
    }
#pragma unroll
    for (int d = 0; d < L::DEPTH; ++d) issue(min(d, units - 1), d);
    asm_wait_vmcnt<L::DEPTH * L::NDMA>();
#pragma unroll
    for (int j = 0; j < SK_KB; ++j) {
        asm_pin(xr[j][0]);
        asm_pin(xr[j][1]);
        if (j >= cnt) xr[j][0] = xr[j][1] = u32x4{0u, 0u, 0u, 0u};   // blocks past the wave's range
    }
#pragma unroll
    for (int j = 0; j < SK_KB; ++j) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[e] = __uint_as_float(xodd ? xr[j][1][e] : xr[j][0][e]);
            x[4 + e] = __uint_as_float(xodd ? xr[j][0][e] : xr[j][1][e]);
        }
        split3(x, xp[j][0], xp[j][1], xp[j][2]);
        sx[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (Q4) {
            const u32x4 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};   // bf16 1.0 pairs
            sx[j] = mfma16(xp[j][0], ones, sx[j]);
            sx[j] = mfma16(xp[j][1], ones, sx[j]);
            sx[j] = mfma16(xp[j][2], ones, sx[j]);
#pragma unroll
            for (int i = 0; i < 4; ++i) sx[j][i] *= -8.0f;
        }
    }
    if (cnt == 0) asm_wait_vmcnt<0>();        // nothing waits for this wave's repeats below
    block_sync();                             // the scales of every wave have landed

    // a lane's scales: row l16 of the row group, from the wave's first
    // block; its codes of block j: a dword (Q4_0) or two (Q8_0)
    const uint32_t s_lane = scale_base + (uint32_t)(l16 * SK_SCALE_DW * 4 + 2 * (((l16 * nb + cb0) & 1) + wave * per));
    const uint32_t c_lane = ring + (uint32_t)(l16 * L::CB + 16 * L::piece(Q4 ? 0 : q >> 1, l16) +
                                              (Q4 ? 4 * q : 8 * (q & 1)));
    // extra: epilogue loads of the wave issued after this row group's codes
    auto unit = [&](int u, int slot, bool extra) {
        if (cnt == 0) return;
        if (u + L::DEPTH > units) asm_wait_vmcnt<0>();
        else if (extra) asm_wait_vmcnt<(L::DEPTH - 1) * L::NDMA + SK_EP_LOADS>();
        else asm_wait_vmcnt<(L::DEPTH - 1) * L::NDMA>();
        const uint32_t src = c_lane + (uint32_t)(slot * L::SLOT);
        const uint32_t ssrc = s_lane + (uint32_t)(u * SK_SCALE_ROWS);
        u32x2 raw[SK_KB];
        uint32_t dh[SK_KB];
        static_for<SK_KB>([&](auto J) {
            constexpr int j = decltype(J)::value;
            // a row's slot is aligned to its size: XOR moves between pieces
            if constexpr (Q4) raw[j][0] = asm_lds_read_b32(src ^ (uint32_t)(16 * j));
            else raw[j] = asm_lds_read_b64(src ^ (uint32_t)(32 * j));
            dh[j] = asm_lds_read_u16<2 * j>(ssrc);
        });
        asm_wait_lgkmcnt<0>();
#pragma unroll
        for (int j = 0; j < SK_KB; ++j) {
            asm_pin(raw[j]);
            asm_pin(dh[j]);
        }
        if (u + L::DEPTH < units) issue(u + L::DEPTH, slot);
        // four blocks at a time (those past the wave's range: X and d are zero)
#pragma unroll
        for (int h = 0; h < SK_KB; h += 4) {
            if (h >= cnt) break;
            f32x4 p[4];
            u32x4 w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = codes_to_bf16<Q4>(raw[h + j]);
#pragma unroll
            for (int j = 0; j < 4; ++j) p[j] = mfma16(xp[h + j][0], w[j], sx[h + j]);
#pragma unroll
            for (int j = 0; j < 4; ++j) p[j] = mfma16(xp[h + j][1], w[j], p[j]);
#pragma unroll
            for (int j = 0; j < 4; ++j) p[j] = mfma16(xp[h + j][2], w[j], p[j]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float d = h + j < cnt ? f16_bits_to_f32((uint16_t)dh[h + j]) : 0.0f;
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i] = __builtin_fmaf(d, p[j][i], acc[i]);
            }
        }
    };

    int slot = 0;
    for (int ub = 0; ub < units; ub += SK_BATCH) {
        const int un = min(SK_BATCH, units - ub);
        for (int k = 0; k < un; ++k) {
            acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            unit(ub + k, slot, ep && ub > 0 && k < L::DEPTH && ub + duty < units);
            slot = slot + 1 == L::DEPTH ? 0 : slot + 1;
            *(reinterpret_cast<f32x4*>(part) + (k * SK_WAVES + wave) * 64 + lane) = acc;
        }
        block_sync();
        if (duty < un && 8 * (wave & 1) < M) {
            const int u = ub + duty, n = n0 + 16 * u + l16;
            const float* from = part + duty * SK_WAVES * 256 + ((wave & 1) * 32 + l16) * 4 + q;
            float sum[2] = {from[0], from[64]};
#pragma unroll
            for (int w = 1; w < SK_WAVES; ++w) {        // in wave order
                sum[0] += from[w * 256];
                sum[1] += from[w * 256 + 64];
            }
            if (ep) {
                // requested before the codes of the batch's refills, of
                // which a wave without blocks has none
                if (cnt > 0 && ub + SK_BATCH + L::DEPTH <= units) asm_wait_vmcnt<SK_BATCH * L::NDMA>();
                else asm_wait_vmcnt<0>();
                float v[SK_EP_LOADS];
#pragma unroll
                for (int i = 0; i < SK_EP_LOADS; ++i)
                    v[i] = __uint_as_float(asm_lds_read_b32(ep_base + (uint32_t)(256 * i + 4 * lane)));
                asm_wait_lgkmcnt<0>();
#pragma unroll
                for (int i = 0; i < SK_EP_LOADS; ++i) asm_pin(v[i]);
                if (u + SK_BATCH < units) issue_ep(u + SK_BATCH);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    float o = sum[i];
                    if (P.ep.bias) o += v[0];
                    if (P.ep.act == 1) o = gelu_tanh(o);
                    else if (P.ep.act == 2) o = silu(o);
                    if (P.ep.mul) o *= v[1 + i];
                    if (P.ep.res) o += v[3 + i];
                    sum[i] = o;
                }
            }
            float* out = cpart ? cpart + (int64_t)c * M * N : P.Y;
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if (om + 4 * i < M && n < N) out[(int64_t)(om + 4 * i) * N + n] = sum[i];
        }
        if (ub + SK_BATCH < units) block_sync();   // the sums are read before the next batch's are written
    }
}

// Adds the chunks of the problems that were split over K, in chunk order.
__global__ __launch_bounds__(256) void skinny_reduce_kernel(const SkinnyGroup g) {
    const SkinnyProblem& P = g.p[blockIdx.y];
    const int64_t mn = (int64_t)g.M * P.N;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (!P.part || i >= mn) return;
    float sum = P.part[i];
    for (int c = 1; c < P.chunks; ++c) sum += P.part[c * mn + i];
    P.Y[i] = P.ep_on ? apply_epilogue(P.ep, sum, i, i % P.N) : sum;
}

static int skinny_chunks(int K) { return (K / 32 + SK_CHUNK - 1) / SK_CHUNK; }

// How a launch of the X-stationary kernel is dealt out: row groups per workgroup,
// workgroups, and rounds of one workgroup per CU (the fewest, of the fewest row
// groups each).
struct SkinnyDeal {
    int rows;
    int64_t blocks, rounds;
};
static SkinnyDeal skinny_deal(int count, const mvlm_weight* const* ws, int num_cus) {
    int64_t units = 0;
    for (int i = 0; i < count; ++i) units += (int64_t)((ws[i]->N + 15) / 16) * skinny_chunks(ws[i]->K);
    for (int64_t rounds = (units + (int64_t)num_cus * SK_MAX_RG - 1) / ((int64_t)num_cus * SK_MAX_RG);; ++rounds)
        for (int rows = (int)((units + num_cus * rounds - 1) / (num_cus * rounds)); rows <= SK_MAX_RG; ++rows) {
            int64_t blocks = 0;
            for (int i = 0; i < count; ++i)
                blocks += (int64_t)(((ws[i]->N + 15) / 16 + rows - 1) / rows) * skinny_chunks(ws[i]->K);
            if (blocks <= num_cus * rounds) return {rows, blocks, rounds};
        }
}

// Whether the X-stationary kernel takes a launch: where its modelled time is no
// longer than that of the kernel that walks K.  Bringing X in once (2.2 us, and a
// second launch of 2.5 us where rows are cut) pays for launches of many row
// groups or long rows; the other kernel is ahead on few row groups, on short rows
// and on rows little longer than a whole number of chunks.  Both measured at
// M = 16, Q8_0: 2048 x 64 4.6 us (K walked) and 7.0 (X kept), 8192 x 768 7.1 and
// 9.2, 8192 x 3072 12.1 and 15.0; 51200 x 2048 38.7 and 27.3, 2048 x 8192 16.6 and
// 14.0, 32000 x 1024 15.4 and 14.3.  The costs are fitted to the times of both
// over 2700 launches (N 64 .. 51200, K 64 .. 11008, M 5 .. 16, single and
// grouped): the choice is 0.4% from the faster one on average, and more than 6%
// from it in 2.5% of them.  MVLM_SKINNY_FORM=x or k forces one (tests, tuning; read
// at every launch).
static bool skinny_keeps_x(int M, int count, const mvlm_weight* const* ws, int num_cus) {
    if (const char* force = std::getenv("MVLM_SKINNY_FORM")) return force[0] == 'x';
    for (int i = 0; i < count; ++i)
        if (ws[i]->K > 16384) return true;   // beyond the fit (Q8_0 8192 x 32768: 72 us, 81 with K walked; 2048 rows 26 and 38)
    struct Cost {
        double launch, row_group, block, row, cut, partial, round;
    };
    constexpr Cost kQ8{5.7, 0.51, 0.0171, 0.092, 2.5, 2.0, 5.1}, kQ4{5.5, 0.49, 0.0116, 0.084, 2.3, 2.3, 4.2};
    const Cost& c = ws[0]->dtype == MVLM_Q4_0 ? kQ4 : kQ8;
    const SkinnyDeal deal = skinny_deal(count, ws, num_cus);
    double units = 0, blocks = 0, parts = 0;   // row groups times chunks, their blocks of K, 10^6 partial sums
    for (int i = 0; i < count; ++i) {
        const int chunks = skinny_chunks(ws[i]->K), nb = ws[i]->K / 32;
        const double u = (double)((ws[i]->N + 15) / 16) * chunks;
        units += u;
        blocks += u * ((nb + chunks - 1) / chunks);
        if (chunks > 1) parts += 1e-6 * M * ws[i]->N * chunks;
    }
    const double busy = std::min((double)deal.blocks / num_cus, (double)deal.rounds) * deal.rows;
    const double us = c.launch + c.row_group * deal.rounds * deal.rows + c.block * busy * (blocks / units) + c.row * M +
                      (parts > 0 ? c.cut + c.partial * parts : 0.0) + c.round * (deal.rounds - 1);
    return us < 1.02 * skinny_kwalk_us(M, count, ws, num_cus);
}

static size_t skinny_partial_bytes(int M, int count, const mvlm_weight* const* ws) {
    size_t bytes = 0;
    for (int i = 0; i < count; ++i) {
        const int chunks = skinny_chunks(ws[i]->K);
        if (chunks > 1) bytes += (size_t)chunks * M * ws[i]->N * sizeof(float);
    }
    return bytes;
}

size_t skinny_workspace_bytes(int M, int count, const mvlm_weight* const* ws, int num_cus) {
    return skinny_keeps_x(M, count, ws, num_cus > 0 ? num_cus : 256) ? skinny_partial_bytes(M, count, ws) : 0;
}

// Which launches are taken: K a multiple of 32, codes and X within 32-bit
// buffer offsets, and rows whose scales fit the LDS of the kernel that walks K,
// which any launch may come down to (it needs no workspace).
bool skinny_supported(int count, const mvlm_weight* const* ws, int num_cus) {
    for (int i = 0; i < count; ++i) {
        const mvlm_weight* w = ws[i];
        if (!is_quant(w->dtype) || w->K % 32 != 0) return false;
        if (w->bytes > 0x7FFFFFFF || (int64_t)16 * w->K * 4 > 0x7FFFFFFF) return false;   // 32-bit buffer offsets
    }
    return skinny_kwalk_fits(count, ws, num_cus > 0 ? num_cus : 256);
}

template <bool Q4>
static hipError_t launch_skinny(hipStream_t s, SkinnyGroup& g, const SkinnyDeal& deal) {
    constexpr auto kernel = gemm_skinny_kernel<Q4>;
    constexpr int lds = SkinnyLayout<Q4>::LDS;
    if (const hipError_t e = allow_dynamic_lds<kernel>(lds); e != hipSuccess) return e;
    int64_t most = 0, begin = 0;   // outputs of the largest problem cut over K; workgroups dealt out
    for (int i = 0; i < g.count; ++i) {
        SkinnyProblem& p = g.p[i];
        p.rows = deal.rows;
        g.block_begin[i] = (int)begin;
        begin += (int64_t)(((p.N + 15) / 16 + p.rows - 1) / p.rows) * p.chunks;
        if (p.part) most = std::max(most, (int64_t)g.M * p.N);
    }
    const dim3 grid((unsigned)deal.blocks), block(64 * SK_WAVES);
    if (most == 0) {
        launch_kernel(kernel, grid, block, (uint32_t)lds, s, g);
        return hipGetLastError();
    }
    launch_kernel_part(LaunchPart::First, kernel, grid, block, (uint32_t)lds, s, g);
    launch_kernel_part(LaunchPart::Last, skinny_reduce_kernel, dim3((unsigned)((most + 255) / 256), (unsigned)g.count),
                       dim3(256), 0, s, g);
    return hipGetLastError();
}

hipError_t launch_gemm_skinny_group(hipStream_t s, int M, int count, const float* const* Xs,
                                    const mvlm_weight* const* ws, float* const* Ys, int num_cus,
                                    const Epilogue* eps, void* workspace, size_t workspace_bytes) {
    if (M < 1 || M > 16 || count < 1 || count > SKINNY_MAX_GROUP) return hipErrorInvalidValue;
    if (num_cus <= 0) num_cus = 256;
    for (int i = 0; i < count; ++i)
        if (ws[i]->K % 32 != 0 || !is_quant(ws[i]->dtype) || ws[i]->dtype != ws[0]->dtype) return hipErrorInvalidValue;
    const size_t need = skinny_partial_bytes(M, count, ws);
    if ((need > 0 && (!workspace || workspace_bytes < need)) || !skinny_keeps_x(M, count, ws, num_cus))
        return launch_skinny_kwalk(s, M, count, Xs, ws, Ys, num_cus, eps);
    float* part = (float*)workspace;
    SkinnyGroup g{};
    g.count = count;
    g.M = M;
    for (int i = 0; i < count; ++i) {
        const mvlm_weight* W = ws[i];
        SkinnyProblem& p = g.p[i];
        p.X = Xs[i];
        p.codes = (const uint8_t*)W->data;
        p.scales = (const uint16_t*)W->scales;
        p.Y = Ys[i];
        p.ld = (uint32_t)W->ld;
        p.N = W->N;
        p.nb = W->K / 32;
        p.chunks = skinny_chunks(W->K);
        p.chunk_blocks = (W->K / 32 + p.chunks - 1) / p.chunks;
        p.chunk_div = (uint32_t)((((uint64_t)1 << 32) + p.chunks - 1) / p.chunks);   // (not used for one chunk)
        if (p.chunks > 1) {
            p.part = part;
            part += (size_t)p.chunks * M * W->N;
        }
        if (eps && eps[i].any()) {
            p.ep = eps[i];
            p.ep_on = 1;
        }
    }
    const SkinnyDeal deal = skinny_deal(count, ws, num_cus);
    return ws[0]->dtype == MVLM_Q4_0 ? launch_skinny<true>(s, g, deal) : launch_skinny<false>(s, g, deal);
}

}  // namespace mvlm
