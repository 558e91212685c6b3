// Batched ternary GEMM for gfx950 (MI355X): Y[m][i] = sum_j W[i][j] X[m][j] for M tokens, exact int32, on the matrix
// cores (v_mfma_i32_32x32x32_i8).
//
// The reference has no multi-token kernel: its prefill runs one GEMV per token (quintrit-runtime/src/engine.rs:625-631),
// so the definition is M independent GEMVs (quintrit-core/src/simd/avx512.rs:1526-1626), and the result must equal
// them bit for bit. Weights stay in the velurex device layout of the GEMV (1.60 bits per weight in HBM) and are
// decoded to int8 trits in registers right before the matrix-core instruction; activations are staged once per call
// in the order of the MFMA B operand.
//
// MFMA operands (v_mfma_i32_32x32x32_i8): lane l supplies 16 int8 of row l % 32 of A (a weight row) and of column
// l % 32 of B (a token); lanes l and l + 32 hold the two halves of the 32-deep K block, and C register r of lane l is
// row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32. Any order of K works as long as A and B use the same one.
//
// K order. A K step is two 16-byte chunks of a weight row: 32 byte-columns x 5 planes = 160 trits = five 32-deep MFMA
// blocks. Lane (i, s) (i = row in the 32-row block, s = lane / 32) holds chunk 2 ks + s of its row in one 16-byte load.
// Block m < 4 takes dword m of that chunk: bytes 4m .. 4m+3, planes 0..3 (t0..t3 as int8, one LDS table lookup per
// byte). Block 4 takes plane 4 of all 16 bytes: t4 = floor(B / 84) - 1 per byte from carry-free byte arithmetic
// (t4_bytes). The activation staging writes X in exactly this order, so A and B pair every weight with its
// activation.
//
// Two kernels: up to 32 tokens gemm_small_kernel (latency: all of a slice's weights in flight at once), beyond that
// gemm_kernel (a tile of row blocks x token groups, pipelined). Long K is split into slices whose int32 partial sums a
// second kernel adds.
#include "vx_gemv_core.h"
#include "vx_internal.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace vx {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4g __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) const u32x4g g_u4g;
typedef u32x4g u32x4u __attribute__((aligned(1)));  // 16- and 4-byte loads at any address
typedef uint32_t u32u __attribute__((aligned(1)));

// t0..t3 of every byte as int8 in a dword (trits03_word: non-values give zero trits, pack.rs:41-58), built at compile
// time; a workgroup copies it into its LDS table with loads.
__constant__ TritTable g_gemm_trits = make_trit_table();

constexpr uint32_t kStepChunks = 2;  // 16-byte chunks per K step
constexpr uint32_t kZeroWord = 0x7d7d7d7du;  // four bytes of five zero trits

// ---- activation staging --------------------------------------------------------------------------------------------

// Staging: thread (token m, pair) writes the five B fragments of K step ks = pair / 2, half hs = pair % 2 of token m:
// xs[ks][kb][tg][lane] (tg = m / 32, lane = (m % 32) + 32 hs) for K blocks kb = 0..4, in the K order of the weight
// decode (column_activation_index, pack.rs:230-237). In a whole 160-trit block (ks < cols / 160) the step is the 160
// activations of block ks and half hs covers byte-columns 16 hs .. 16 hs + 15: K block kb < 4 takes, for byte-column
// 16 hs + 4 kb + d, its activations of planes 0..3, a(160 ks + 32 e + 16 hs + 4 kb + d), e = 0..3: dword kb of the
// four 16-byte loads at 160 ks + 32 e + 16 hs (at any alignment), transposed 4 x 4 bytes with v_perm; K block 4 takes
// plane 4 of the 16 byte-columns, the 16 bytes at 160 ks + 128 + 16 hs as they are. The packed tail takes the per-byte
// gather. Workgroup (pair block, token group): lane j of each 32-thread row is token 32 tg + j and the rows are
// kStageRows consecutive pairs, so the 32 tokens of a row write one contiguous 512-byte run per K block.
constexpr uint32_t kStageRows = 8;  // pairs per staging workgroup (256 threads)

// The five fragments of half hs of a whole block from its pieces X[e] = activations 32 e + 16 hs .. + 15 (plane e of the
// 16 byte-columns): K block kb < 4 the 4 x 4 byte transpose of dword kb of planes 0..3, K block 4 plane 4 as it is.
__device__ __forceinline__ void block_fragments(const u32x4g (&X)[5], u32x4g (&o)[5]) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        auto dw = [&](const u32x4g& v) { return kb == 0 ? v.x : (kb == 1 ? v.y : (kb == 2 ? v.z : v.w)); };
        const uint32_t a0 = dw(X[0]), a1 = dw(X[1]), a2 = dw(X[2]), a3 = dw(X[3]);
        const uint32_t lo01 = __builtin_amdgcn_perm(a1, a0, 0x05010400u), hi01 = __builtin_amdgcn_perm(a1, a0, 0x07030602u);
        const uint32_t lo23 = __builtin_amdgcn_perm(a3, a2, 0x05010400u), hi23 = __builtin_amdgcn_perm(a3, a2, 0x07030602u);
        o[kb] = u32x4g{__builtin_amdgcn_perm(lo23, lo01, 0x05040100u), __builtin_amdgcn_perm(lo23, lo01, 0x07060302u),
                           __builtin_amdgcn_perm(hi23, hi01, 0x05040100u), __builtin_amdgcn_perm(hi23, hi01, 0x07060302u)};
    }
    o[4] = X[4];
}

// The same for a half of the packed tail, X its 80 consecutive activations: byte-column k holds activations 5 k .. 5 k +
// 4, so dword d of K block kb < 4 is the four bytes from 5 (4 kb + d) on, of K block 4 bytes 5 (4 d + e) + 4, e = 0..3.
__device__ __forceinline__ void tail_fragments(const u32x4g (&X)[5], u32x4g (&o)[5]) {
    const uint32_t D[21] = {X[0].x, X[0].y, X[0].z, X[0].w, X[1].x, X[1].y, X[1].z, X[1].w, X[2].x, X[2].y, X[2].z,
                            X[2].w, X[3].x, X[3].y, X[3].z, X[3].w, X[4].x, X[4].y, X[4].z, X[4].w, 0u};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        uint32_t v[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const int b = 20 * kb + 5 * d;
            v[d] = __builtin_amdgcn_alignbyte(D[b / 4 + 1], D[b / 4], b % 4);
        }
        o[kb] = u32x4g{v[0], v[1], v[2], v[3]};
    }
    uint32_t v[4];
#pragma unroll
    for (int d = 0; d < 4; ++d)
        v[d] = __builtin_amdgcn_perm(D[5 * d + 2], D[5 * d + 1], 0x0c0c0500u) |
               __builtin_amdgcn_perm(D[5 * d + 4], D[5 * d + 3], 0x07020c0cu);
    o[4] = u32x4g{v[0], v[1], v[2], v[3]};
}

__global__ __launch_bounds__(256) void gemm_stage_kernel(const int8_t* __restrict__ x, uint32_t ldx, uint32_t n_tg,
                                                         uint32_t cols, uint32_t n_ksteps,
                                                         u32x4g* __restrict__ xs, uint32_t M) {
    const uint32_t tid = threadIdx.x, j = tid & 31u;
    const uint32_t pair = blockIdx.x * kStageRows + (tid >> 5), ks = pair >> 1, hs = pair & 1u;
    const uint32_t tg = blockIdx.y, m = tg * 32u + j;
    // B fragments of tokens past M (the rest of the last 32-token group) are left as they are: they only reach C
    // columns that are never stored.
    if (ks >= n_ksteps || m >= M) return;
    const int8_t* xr = x + static_cast<size_t>(m) * ldx;
    u32x4g o[5];
    if (ks < cols / 160u) {
        const int8_t* blk = xr + ks * 160u + 16u * hs;
        u32x4g X[5];
#pragma unroll
        for (int e = 0; e < 5; ++e) X[e] = *reinterpret_cast<const u32x4u*>(blk + 32 * e);
        block_fragments(X, o);
    } else {
        // the packed tail: byte-column 16 hs + k of the step (k < 16), activation p is 160 ks + 5 (16 hs + k) + p
        // (column_activation_index); past the row (and in the tail's padding columns, whose indices are all >= cols) zero
        auto act = [&](uint32_t k, uint32_t p) -> uint32_t {
            const uint32_t idx = ks * 160u + 5u * (16u * hs + k) + p;
            return idx < cols ? static_cast<uint32_t>(static_cast<uint8_t>(xr[idx])) : 0u;
        };
#pragma unroll
        for (uint32_t kb = 0; kb < 5; ++kb) {
            uint32_t w[4];
#pragma unroll
            for (uint32_t d = 0; d < 4; ++d) {
                uint32_t v = 0;
#pragma unroll
                for (uint32_t e = 0; e < 4; ++e) v |= (kb < 4 ? act(4u * kb + d, e) : act(4u * d + e, 4u)) << (8 * e);
                w[d] = v;
            }
            o[kb] = u32x4g{w[0], w[1], w[2], w[3]};
        }
    }
#pragma unroll
    for (uint32_t kb = 0; kb < 5; ++kb) xs[(static_cast<size_t>(ks * 5u + kb) * n_tg + tg) * 64u + j + 32u * hs] = o[kb];
}

// ---- GEMM -------------------------------------------------------------------------------------------------------------

// One matrix of a call: up to kGemmSubs matrices with the same columns share a launch, their tiles (and 32-row blocks)
// concatenated. Its tiles are tiles tile0 .. tile0 + n_tiles - 1 of the call, its rows rows row0 .. row0 + rows_p - 1 of
// the slice sums.
constexpr int kGemmSubs = 3;
struct GemmMat {
    const uint8_t* w;
    int32_t* y;
    uint32_t ldy, rows, rows_p, n_tiles, tile0, row0;
};

struct GemmArgs {
    GemmMat sub[kGemmSubs];
    uint32_t n_sub;
    const int8_t* x;     // raw activations, M rows of ldx
    const u32x4g* xs;     // staged activations (gemm_kernel without RAW)
    int32_t* part;       // [kslices][M][rows_p] slice sums (kslices > 1)
    uint32_t ldx, rows_p, cols, n_tiles, n_chunks, n_ksteps, M, n_tg, kslices;  // rows_p, n_tiles: of all the matrices
    uint32_t steps;      // K steps per slice
    uint32_t n_rg, n_tt; // gemm_kernel: row groups of 4 R blocks, token tiles of T groups
};

// More than 32 tokens. A workgroup of 4 waves takes 4 R consecutive 32-row blocks (wave w blocks R w .. R w + R - 1 of
// them), T groups of 32 tokens and the K steps of a slice. The A fragments are decoded in registers, once for all T
// groups, the B fragments of a K step are in LDS for all waves.
//
// Everything is pipelined in units of one K block (R T matrix products): while the products of K block kb run, the
// wave looks up the trits and reads the B fragments of K block kb + 1 into the other of two register sets. The weights
// are requested three K steps ahead, the activations of step k + 3 during step k and written to LDS as fragments a step
// before their use (two buffers, one barrier per step, placed where the last reads of the step have been issued). With
// 8-wave workgroups that decoded a whole K step behind the barrier before its products, the matrix pipe idled through
// every decode. 2560 x 2560 x 512 tokens 30.4 -> 15.9 us per call, 23040 x 3072 x 128 38 -> 23.7, 6913 x 2563 x 100 35.8 ->
// 15.4 (staging launch included), 23040 x 3072 x 512 56.9 -> 45.1 (1.61 POP/s; a plain int8 library product of 8192^3
// reaches 2.1 on this card). 3072 x 23040 x 512, whose 31 MB of slice sums are written and read back, gained nothing (65 to
// 69 us before and after).
//
// What bounds it: instruction issue. A wave issues an instruction about every 7 cycles, matrix products included, and a
// K step of one wave is 5 R T products of 32 cycles beside 16 R lookups with their addresses, 36 R byte operations for
// plane 4, 5 T fragment reads and about 60 others: 1.26 us per step at R = 3, T = 4, of which 0.8 are products. At 512
// tokens of 3072-column rows the output (47 MB) and the start of the call take as long as the rest.
//
// RAW (cols in whole 16-byte pieces, at any alignment): the workgroup builds the B fragments from x itself: lane (token,
// half) loads the 80 activations of its half of the K step as five 16-byte pieces and transposes them (in a whole block
// four 4 x 4 byte transposes, in the packed tail of the row, whose byte-columns hold five consecutive activations, byte
// shifts). Pieces past the row read its last one: the weights there are zero trits; a chunk past the row, whose weights
// repeat the last chunk's, gets zeros. Its scattered loads cost about 0.1 us per step more than those of fragments that
// gemm_stage_kernel or the caller has written (xs); the staging launch costs 4 us where calls follow one another (3072 x
// 3072 x 64 17 against 12 us per call, 23040 x 3072 x 128 25.5 against 23.4).
//
// LDS: the trit table (row B: 32 copies of byte B's entry in the first 128 bytes of a 256-byte row; lane l reads copy
// l % 32, conflict-free because LDS serves a wave in two 32-lane halves), and in the second halves of its rows the two
// buffers of fragments, 8 rows of 128 bytes each: 80 KiB for four token groups, so that two workgroups fit a CU where
// their registers do.
//
// Workgroups: the list (row group, K slice, token tile), token tiles fastest, in eight equal parts, one per XCD
// (blockIdx.x mod 8): the token tiles that read the same weights share an L2, and every XCD has work however few row
// groups there are. (With whole row groups per XCD, row group mod 8, most of the card idled below 8 of them and parts of
// it at 9 to 15: 300 x 23040 x 512 36.1 -> 20.2 us, 3072 x 23040 x 64 26.4 -> 21.1, 40 x 3072 x 512 20.6 -> 9.8.) Row
// groups in whole eights keep that assignment within the list: neighbouring row groups on one XCD instead took 14.5 us
// against 11.8 at 8192 x 3072 x 33 in calls repeated with one workspace. (Only there: 8192 x 3072 x 64 takes 15.6 us with
// one workspace, 12.9 with another for each call, in either order, and the L2 misses are alike. Probably this kernel's
// stores wait for lines that the finish kernel of the call before read on another XCD; not observed directly.)
template <int T, int R, bool RAW>
__global__ __launch_bounds__(256, T * R >= 8 ? 1 : 2) void gemm_kernel(GemmArgs a) {
    constexpr uint32_t kFrags = 5u * T;                 // B fragments of a K step
    constexpr uint32_t kXPer = RAW ? 5u : (kFrags + 3u) / 4u;  // 16-byte loads of activations per thread and step
    constexpr int kReads = 4 * R + T, kEarly = (R * T + 1) / 2;  // the LDS reads of a K block follow its first products
    constexpr uint32_t kLdsRows = 2u * kFrags * 8u > 256u ? 2u * kFrags * 8u : 256u;
    __shared__ __align__(256) uint32_t tab[kLdsRows * 64u];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, half = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t total = a.n_rg * a.kslices * a.n_tt, item = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (item >= total) return;
    uint32_t tt = 0, kz = 0, rg = item;  // (divisions only where they are needed: they cost the smallest calls 0.25 us)
    if (a.n_tt > 1u) tt = rg % a.n_tt, rg /= a.n_tt;
    if (a.kslices > 1u) kz = rg % a.kslices, rg /= a.kslices;
    if (a.n_rg % 8u == 0u && a.n_rg > 8u) rg = rg % (a.n_rg >> 3) * 8u + rg / (a.n_rg >> 3);
    const uint32_t ks0 = kz * a.steps, ks1 = min(ks0 + a.steps, a.n_ksteps), last = ks1 - 1u;
    const uint32_t blk0 = (rg * 4u + wave) * R, n_blk = 2u * a.n_tiles;

    // The wave's blocks: block 2 t + h is rows 32 h .. of tile t of its matrix (16 bytes a row per chunk, the chunks of a
    // tile T_g KiB apart in its tile group). A block past the call reads the last one and stores nothing.
    auto sub_of = [&](uint32_t tile) -> const GemmMat& {
        return a.n_sub > 2u && tile >= a.sub[2].tile0 ? a.sub[2] : (a.n_sub > 1u && tile >= a.sub[1].tile0 ? a.sub[1] : a.sub[0]);
    };
    // Addresses are a scalar base, advanced by each load until the slice's last step, and a 32-bit lane offset. A chunk
    // past the row (odd n_chunks) repeats the one before it: its activations are zero.
    const uint8_t* wp[R];
    uint32_t cstride[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t blk = min(blk0 + r, n_blk - 1u);
        const GemmMat& sb = sub_of(blk >> 1);
        const uint32_t tile = (blk >> 1) - sb.tile0, grp = tile / kTileGroup, t16 = tile - grp * kTileGroup;
        const uint32_t Tg = min(static_cast<uint32_t>(kTileGroup), sb.n_tiles - grp * kTileGroup);
        cstride[r] = Tg * 1024u;
        wp[r] = sb.w + (static_cast<size_t>(grp) * kTileGroup * a.n_chunks + t16) * 1024u + (blk & 1u) * 512u +
                static_cast<size_t>(ks0 * kStepChunks) * cstride[r];
    }
    const uint32_t woff = (lane & 31u) * 16u;
    auto load_w = [&](uint32_t ks, u32x4g (&wv)[R]) __attribute__((always_inline)) {  // step min(ks, last), in order
        const bool two = min(ks, last) * kStepChunks + 1u < a.n_chunks;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            wv[r] = *(g_u4g*)(wp[r] + (woff + (two && half != 0 ? cstride[r] : 0u)));
            wp[r] += ks < last ? kStepChunks * cstride[r] : 0u;
        }
    };

    char* const lds = reinterpret_cast<char*>(tab);
    const uint32_t frag_lane = (lane >> 3) * 256u + 128u + (lane & 7u) * 16u;  // + 2048 per fragment
    const auto frag_at = [&](uint32_t buf, uint32_t f) { return reinterpret_cast<u32x4g*>(lds + frag_lane + (buf * kFrags + f) * 2048u); };
    // RAW: wave w < T builds the fragments of token group w, lane (j, hs) token j's half hs; the other waves load one
    // address and store to spare fragments (a branch around loads would make every wait after it one for all loads).
    // Otherwise the fragments f = kb T + g are copied, wave w those with f % 4 = w (one past the last
    // repeats it, and one of a token group past M the last group's: it reaches outputs that are never stored).
    static_assert(2u * kFrags + 5u * (4u - T) <= kLdsRows / 8u, "spare fragments of the waves without a token group");
    const uint32_t hs = half, full = a.cols / 160u;
    const uint32_t xrow_m = wave < T ? min((tt * T + wave) * 32u + (lane & 31u), a.M - 1u) : 0u;
    const int8_t* xrow = a.x + static_cast<size_t>(xrow_m) * a.ldx;
    const uint32_t xhs = wave < T ? hs : 0u;
    const auto raw_frag = [&](uint32_t buf, uint32_t kb) {
        return frag_at(0u, wave < T ? buf * kFrags + kb * T + wave : 2u * kFrags + (wave - T) * 5u + kb);
    };
    const u32x4g* xp[kXPer];
    if constexpr (!RAW) {
#pragma unroll
        for (uint32_t i = 0; i < kXPer; ++i) {
            const uint32_t f = min(wave + 4u * i, kFrags - 1u);
            xp[i] = a.xs + (static_cast<size_t>(ks0 * 5u + f / T) * a.n_tg + min(tt * T + f % T, a.n_tg - 1u)) * 64u;
        }
    }
    const uint32_t xstep = 5u * a.n_tg * 64u;
    u32x4g X[2][kXPer];
    auto load_x = [&](uint32_t ks, u32x4g (&x)[kXPer]) __attribute__((always_inline)) {  // step min(ks, last), in order
        if constexpr (RAW) {
            const uint32_t k = min(ks, last), base = k * 160u + xhs * (k < full ? 16u : 80u), step = k < full ? 32u : 16u;
#pragma unroll
            for (uint32_t i = 0; i < kXPer; ++i) x[i] = *reinterpret_cast<const u32x4u*>(xrow + min(base + i * step, a.cols - 16u));
        } else {
#pragma unroll
            for (uint32_t i = 0; i < kXPer; ++i) {
                x[i] = *(g_u4g*)(xp[i] + lane);
                xp[i] += ks < last ? xstep : 0u;
            }
        }
    };
    auto store_x = [&](uint32_t buf, const u32x4g (&x)[kXPer]) __attribute__((always_inline)) {
        if constexpr (RAW) {
            u32x4g o[5];
            block_fragments(x, o);
#pragma unroll
            for (uint32_t kb = 0; kb < 5; ++kb) *raw_frag(buf, kb) = o[kb];
        } else {
#pragma unroll
            for (uint32_t i = 0; i < kXPer; ++i) *frag_at(buf, min(wave + 4u * i, kFrags - 1u)) = x[i];
        }
    };
    // RAW: the fragments of step ks in the packed tail, written over what store_x made of them
    auto store_tail = [&](uint32_t ks, uint32_t buf, const u32x4g (&x)[kXPer]) __attribute__((always_inline)) {
        if constexpr (RAW) {
            u32x4g o[5];
            tail_fragments(x, o);
            const bool none = ks * kStepChunks + hs >= a.n_chunks;
#pragma unroll
            for (uint32_t kb = 0; kb < 5; ++kb) *raw_frag(buf, kb) = none ? u32x4g{0u, 0u, 0u, 0u} : o[kb];
        }
    };
    const uint32_t lane_off = (lane & 31u) * 4u;
    // the A fragments of K block kb < 4: t0..t3 of the four bytes of dword kb
    auto dword = [](const u32x4g& v, int k) { return k == 0 ? v.x : (k == 1 ? v.y : (k == 2 ? v.z : v.w)); };
    auto decode = [&](int kb, const u32x4g (&w)[R], v4i (&A)[R]) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            int t[4];
#pragma unroll
            for (int b = 0; b < 4; ++b)
                t[b] = *reinterpret_cast<const int*>(lds + __builtin_amdgcn_perm(dword(w[r], kb), lane_off, 0x0c0c0000u | ((4u + b) << 8)));
            A[r] = v4i{t[0], t[1], t[2], t[3]};
        }
    };
    auto read_b = [&](uint32_t kb, uint32_t buf, v4i (&B)[T]) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t g = 0; g < T; ++g)
            B[g] = *reinterpret_cast<const v4i*>(lds + frag_lane + (buf * kFrags + kb * T + g) * 2048u);
    };

    v16i acc[R][T];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int g = 0; g < T; ++g) acc[r][g] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

    u32x4g w[4][R];
    v4i A[2][R], A4[R], B[2][T];
    load_x(ks0, X[0]);
    load_w(ks0, w[0]);
    load_x(ks0 + 1u, X[1]);
    load_w(ks0 + 1u, w[1]);
    load_w(ks0 + 2u, w[2]);
    for (uint32_t i = tid; i < 256u * 8u; i += 256u) {
        const uint32_t e = g_gemm_trits.v[i >> 3];
        *reinterpret_cast<uint4*>(lds + (i >> 3) * 256u + (i & 7u) * 16u) = make_uint4(e, e, e, e);
    }
    store_x(0, X[0]);
    if (RAW && ks0 >= full) store_tail(ks0, 0, X[0]);
    load_x(ks0 + 2u, X[0]);
    __syncthreads();
    decode(0, w[0], A[0]);
    read_b(0, 0, B[0]);

    // Step ks = ks0 + s (mod 4), with weights w[s], fragments in buffer s & 1. The loads are unconditional (indices clamp
    // at the last step) and the loop has no other exit, so that every wait is for its own load.
    auto step = [&](auto sc, uint32_t ks) __attribute__((always_inline)) {
        constexpr uint32_t s = decltype(sc)::value, buf = s & 1u;
        static_for<5>([&](auto kc) __attribute__((always_inline)) {
            constexpr uint32_t kb = decltype(kc)::value, cur = (s + kb) & 1u, nxt = cur ^ 1u;
            if constexpr (kb == 0) load_w(ks + 3u, w[(s + 3u) & 3u]);
            if constexpr (kb == 2) store_x(buf ^ 1u, X[(s + 1u) & 1u]);
            if constexpr (kb == 3) {
                if (RAW && ks + 1u >= full && ks + 1u < ks1) store_tail(ks + 1u, buf ^ 1u, X[(s + 1u) & 1u]);
                load_x(ks + 3u, X[(s + 1u) & 1u]);
            }
            if constexpr (kb < 4) {
                if constexpr (kb < 3) decode(kb + 1, w[s], A[nxt]);
#pragma unroll
                for (int r = 0; r < R; ++r) A4[r][kb] = static_cast<int>(t4_bytes(dword(w[s][r], kb)));
                read_b(kb + 1u, buf, B[nxt]);
            } else {
                __syncthreads();  // the fragments of step ks + 1 are complete, every read of step ks has been made
                decode(0, w[(s + 1u) & 3u], A[nxt]);
                read_b(0, buf ^ 1u, B[nxt]);
            }
#pragma unroll
            for (int g = 0; g < T; ++g)
#pragma unroll
                for (int r = 0; r < R; ++r)
                    acc[r][g] = __builtin_amdgcn_mfma_i32_32x32x32_i8(B[cur][g], kb < 4 ? A[cur][r] : A4[r], acc[r][g], 0, 0, 0);
            // a product, then reads of the next K block and other instructions in its shadow, and nothing of a K block
            // moved into another
#pragma unroll
            for (int i = 0; i < R * T; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                if (i < kEarly) __builtin_amdgcn_sched_group_barrier(0x100, (kReads + kEarly - 1) / kEarly, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    uint32_t ks = ks0;
    for (; ks + 4u <= ks1; ks += 4u) static_for<4>([&](auto sc) __attribute__((always_inline)) { step(sc, ks + sc); });
    if (ks < ks1) step(std::integral_constant<uint32_t, 0>{}, ks);
    if (ks + 1u < ks1) step(std::integral_constant<uint32_t, 1>{}, ks + 1u);
    if (ks + 2u < ks1) step(std::integral_constant<uint32_t, 2>{}, ks + 2u);

    // The product is taken transposed (activations as the first operand): lane l holds row l % 32 of the block and, in
    // register r, token 8 (r / 4) + 4 (l / 32) + r % 4 of the group, so that a store writes 128 consecutive bytes of two
    // tokens. (With the tokens in the lanes each 16-byte store went to a line of its own.)
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t blk = blk0 + r;
        if (blk >= n_blk) break;
        const GemmMat& sb = sub_of(blk >> 1);
        const uint32_t n = blk * 32u - sb.tile0 * 64u + (lane & 31u);
        const bool slices = a.kslices > 1u;
        const uint32_t ld = slices ? a.rows_p : sb.ldy;
        int32_t* out = slices ? a.part + static_cast<size_t>(kz) * a.M * a.rows_p + sb.row0 : sb.y;
        if (!slices && n >= sb.rows) continue;
#pragma unroll
        for (int g = 0; g < T; ++g)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const uint32_t m = (tt * T + g) * 32u + 8u * (e / 4) + 4u * half + (e % 4);
                if (m < a.M) out[static_cast<size_t>(m) * ld + n] = acc[r][g][e];
            }
    }
}

// Y[m][n] = sum over the slices of their sums (block = 256 rows of the call's slice sums, one token).
template <bool G>
__global__ __launch_bounds__(256) void gemm_finish_kernel(GemmArgs a) {
    const uint32_t n = blockIdx.x * 256u + threadIdx.x, m = blockIdx.y;
    const uint32_t j = !G ? 0u : (a.n_sub > 1u && n >= a.sub[1].row0 ? 1u : 0u) + (a.n_sub > 2u && n >= a.sub[2].row0 ? 1u : 0u);
    const GemmMat sb = j == 0u ? a.sub[0] : (j == 1u ? a.sub[1] : a.sub[2]);  // no indexing of the arguments
    const uint32_t ln = n - sb.row0;
    if (n >= a.rows_p || ln >= sb.rows) return;
    const size_t stride = static_cast<size_t>(a.M) * a.rows_p;
    const int32_t* p = a.part + static_cast<size_t>(m) * a.rows_p + n;
    int s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    uint32_t k = 0;
    for (; k + 4 <= a.kslices; k += 4) {
        s0 += p[k * stride];
        s1 += p[(k + 1) * stride];
        s2 += p[(k + 2) * stride];
        s3 += p[(k + 3) * stride];
    }
    for (; k < a.kslices; ++k) s0 += p[k * stride];
    sb.y[static_cast<size_t>(m) * sb.ldy + ln] = (s0 + s1) + (s2 + s3);
}

// ---- one or two token groups: one launch --------------------------------------------------------------------------

// Workgroup (c, kz): W waves, wave w the 64-row tile W c + w, over the K steps of slice kz (at most kSmallSteps), for T
// groups of 32 tokens. G: the call's tiles may belong to several matrices of the same columns (each wave finds its own;
// without G the instance reads only the first). Each thread first loads the activations of its B-fragment tasks (task =
// step, token group, half, token) and the trit table's entries, then each wave loads all its weights of the slice at once
// (2 chunks per K step per lane, every load unconditional: steps past the slice read its last step again), so the wait
// for the activations and the table does not include the weights' latency (loads return in order); the workgroup then
// builds the trit table and the slice's B fragments in LDS (the staging of gemm_stage_kernel, so no staging kernel runs)
// and each wave multiplies with no further barrier. With one slice the wave writes Y; otherwise it stores its slice's
// sums, which gemm_finish_kernel adds. (Gathering them in the kernel instead, each tile's last slice reading the others'
// sums with agent-scope atomic loads after a ticket, was slower: 30-160 us per call at M = 8-32.)
constexpr uint32_t kSmallSteps = 8;  // K steps per slice at most (40 KiB of B fragments per token group in LDS)

template <int T, int W, bool G, bool TOKENS>
__global__ __launch_bounds__(W * 64) void gemm_small_kernel(GemmArgs a) {
    __shared__ uint32_t tab[256 * 64];
    constexpr uint32_t S = kSmallSteps;
    __shared__ uint4 bs[S * 5 * T * 64];
    constexpr uint32_t kTasks = S * T / W;  // B-fragment tasks per thread
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t tile = blockIdx.x * W + wave, kz = blockIdx.y;
    // the wave's matrix (wave-uniform) and its tile there (a tile past the call's tiles falls in the last matrix)
    const uint32_t j = !G ? 0u : (a.n_sub > 1u && tile >= a.sub[1].tile0 ? 1u : 0u) + (a.n_sub > 2u && tile >= a.sub[2].tile0 ? 1u : 0u);
    const GemmMat sb = j == 0u ? a.sub[0] : (j == 1u ? a.sub[1] : a.sub[2]);
    const uint32_t lt = tile - sb.tile0;
    const uint32_t ks0 = kz * a.steps, nst = min(a.steps, a.n_ksteps - ks0);
    const uint32_t half = lane >> 5;

    // The activations of this thread's tasks, loaded before the weights with every load at a valid address (no
    // branch that depends on the thread separates them from the weight loads, and nothing waits for them before the
    // weights are requested). With a block in the row: a whole 160-column block as 5 uint4 (kind 1);
    // when the slice's last step is the partial last block, its task (one per thread, a task holding W / T steps) as
    // the 80 columns of its half (kind 2). Other tasks are read by bytes after the weight loads (kind 0).
    const bool blocks = a.cols >= 160u;  // x holds a block (its rows may have any alignment)
    const bool has_tail = a.cols % 160u != 0u && ks0 + nst == a.n_ksteps;
    u32x4g X[kTasks][5];
    uint32_t kind[kTasks];
#pragma unroll
    for (uint32_t r = 0; r < kTasks; ++r) {
        const uint32_t t = tid + r * W * 64u;
        const uint32_t s = t / (64u * T), rr = t - s * 64u * T, tok = 32u * (rr >> 6) + (rr & 31u), ks = ks0 + s;
        const uint32_t hs = (rr >> 5) & 1u;
        const bool live = s < nst && tok < a.M;
        kind[r] = !live || !blocks ? 0u : (ks < a.cols / 160u ? 1u : 2u);
        if (blocks) {
            const int8_t* blk = (kind[r] == 1u ? a.x + static_cast<size_t>(tok) * a.ldx + ks * 160u : a.x) + 16u * hs;
#pragma unroll
            for (int e = 0; e < 5; ++e) X[r][e] = *reinterpret_cast<const u32x4u*>(blk + 32 * e);
        }
    }
    // kind 2, raw: the words at clamped addresses and the bytes of the word that straddles cols (masked where used).
    // Loaded by every workgroup (from the weights, which are 256-byte aligned, where no partial block is used) so that
    // no branch joins them before the weight loads.
    uint32_t V[20], tb[3];
    {
        const bool use = has_tail && blocks;
        const uint32_t t = tid + (nst - 1u) * T / W * W * 64u;
        const uint32_t s = t / (64u * T), rr = t - s * 64u * T, tok = 32u * (rr >> 6) + (rr & 31u), hs = (rr >> 5) & 1u;
        const int8_t* row = use ? a.x + static_cast<size_t>(tok < a.M ? tok : 0u) * a.ldx : reinterpret_cast<const int8_t*>(sb.w);
        const uint32_t base = use ? (a.n_ksteps - 1u) * 160u + 80u * hs : 0u, lastw = use ? (a.cols - 4u) & ~3u : 0u;
        const uint32_t i0 = use ? a.cols & ~3u : 0u, lastb = use ? a.cols - 1u : 0u;
#pragma unroll
        for (uint32_t d = 0; d < 20; ++d) V[d] = *reinterpret_cast<const u32u*>(row + min(base + 4u * d, lastw));
#pragma unroll
        for (uint32_t e = 0; e < 3; ++e) tb[e] = static_cast<uint8_t>(row[min(i0 + e, lastb)]);
    }

    // the trit table's entries (256 x 8 uint4 stores of 4 copies each)
    constexpr uint32_t kTabPer = 256u * 8u / (W * 64u);
    uint32_t te[kTabPer];
#pragma unroll
    for (uint32_t r = 0; r < kTabPer; ++r) te[r] = g_gemm_trits.v[(tid + r * W * 64u) >> 3];

    // the weights (a tile past the matrix reads the last one)
    const uint32_t ltile = min(lt, sb.n_tiles - 1u);
    const uint32_t grp = ltile / kTileGroup, t16 = ltile - grp * kTileGroup;
    const uint32_t Tg = min(static_cast<uint32_t>(kTileGroup), sb.n_tiles - grp * kTileGroup);
    const uint8_t* wbase = sb.w + (static_cast<size_t>(grp) * kTileGroup * a.n_chunks + t16) * 1024u + (lane & 31u) * 16u;
    u32x4g wv[S][2];
#pragma unroll
    for (uint32_t s = 0; s < S; ++s) {
        const uint32_t q = min((ks0 + min(s, nst - 1u)) * kStepChunks + half, a.n_chunks - 1u);
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
            wv[s][rb] = __builtin_nontemporal_load((g_u4g*)(wbase + static_cast<size_t>(q) * Tg * 1024u + rb * 512u));
    }

#pragma unroll
    for (uint32_t r = 0; r < kTabPer; ++r) {
        const uint32_t i = tid + r * W * 64u;
        *reinterpret_cast<uint4*>(reinterpret_cast<char*>(tab) + (i >> 3) * 256u + (i & 7u) * 16u) =
            make_uint4(te[r], te[r], te[r], te[r]);
    }
    // B fragments of the slice; tokens past M get zeros
#pragma unroll
    for (uint32_t r = 0; r < kTasks; ++r) {
        const uint32_t t = tid + r * W * 64u;
        const uint32_t s = t / (64u * T), rr = t - s * 64u * T, g = rr >> 6, hs = (rr >> 5) & 1u, j = rr & 31u;
        const uint32_t tok = 32u * g + j, ks = ks0 + s;
        if (s >= nst) continue;
        uint4 o[5] = {};
        if (kind[r] == 1u) {
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
                auto dw = [&](const u32x4g& v) { return kb == 0 ? v.x : (kb == 1 ? v.y : (kb == 2 ? v.z : v.w)); };
                const uint32_t a0 = dw(X[r][0]), a1 = dw(X[r][1]), a2 = dw(X[r][2]), a3 = dw(X[r][3]);
                const uint32_t lo01 = __builtin_amdgcn_perm(a1, a0, 0x05010400u), hi01 = __builtin_amdgcn_perm(a1, a0, 0x07030602u);
                const uint32_t lo23 = __builtin_amdgcn_perm(a3, a2, 0x05010400u), hi23 = __builtin_amdgcn_perm(a3, a2, 0x07030602u);
                o[kb] = make_uint4(__builtin_amdgcn_perm(lo23, lo01, 0x05040100u), __builtin_amdgcn_perm(lo23, lo01, 0x07060302u),
                                   __builtin_amdgcn_perm(hi23, hi01, 0x05040100u), __builtin_amdgcn_perm(hi23, hi01, 0x07060302u));
            }
            o[4] = make_uint4(X[r][4].x, X[r][4].y, X[r][4].z, X[r][4].w);
        } else if (kind[r] == 2u) {
            // column ks * 160 + 80 hs + 5 k + p of the partial block is byte 5 k + p of the 80 loaded
            const uint32_t base = ks * 160u + 80u * hs, i0 = a.cols & ~3u;
            auto byte_at = [&](uint32_t i) -> uint32_t {
                const uint32_t c = base + i;
                return c < i0 ? (V[i >> 2] >> (8u * (i & 3u))) & 0xffu : (c < a.cols ? tb[c & 3u] : 0u);
            };
#pragma unroll
            for (uint32_t kb = 0; kb < 5; ++kb) {
                uint32_t w[4];
#pragma unroll
                for (uint32_t d = 0; d < 4; ++d) {
                    uint32_t v = 0;
#pragma unroll
                    for (uint32_t e = 0; e < 4; ++e)
                        v |= byte_at(kb < 4 ? 5u * (4u * kb + d) + e : 5u * (4u * d + e) + 4u) << (8 * e);
                    w[d] = v;
                }
                o[kb] = make_uint4(w[0], w[1], w[2], w[3]);
            }
        } else if (tok < a.M) {
            const int8_t* xr = a.x + static_cast<size_t>(tok) * a.ldx;
            const bool tail = ks >= a.cols / 160u;
            auto act = [&](uint32_t k, uint32_t p) -> uint32_t {
                const uint32_t idx = tail ? ks * 160u + 5u * (16u * hs + k) + p : ks * 160u + 32u * p + 16u * hs + k;
                return idx < a.cols ? static_cast<uint32_t>(static_cast<uint8_t>(xr[idx])) : 0u;
            };
#pragma unroll
            for (uint32_t kb = 0; kb < 5; ++kb) {
                uint32_t w[4];
#pragma unroll
                for (uint32_t d = 0; d < 4; ++d) {
                    uint32_t v = 0;
#pragma unroll
                    for (uint32_t e = 0; e < 4; ++e) v |= (kb < 4 ? act(4u * kb + d, e) : act(4u * d + e, 4u)) << (8 * e);
                    w[d] = v;
                }
                o[kb] = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
#pragma unroll
        for (uint32_t kb = 0; kb < 5; ++kb) bs[((s * 5u + kb) * T + g) * 64u + j + 32u * hs] = o[kb];
    }
    __syncthreads();
    if (tile >= a.n_tiles) return;

    const char* tabb = reinterpret_cast<const char*>(tab);
    const uint32_t lane_off = (lane & 31u) * 4u;
    v16i acc[2][T];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int g = 0; g < T; ++g) acc[rb][g] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (uint32_t s = 0; s < S; ++s) {
        if (s >= nst) break;
        const bool inside = (ks0 + s) * kStepChunks + half < a.n_chunks;
        v4i A[2][5];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            const uint32_t dw[4] = {inside ? wv[s][rb].x : kZeroWord, inside ? wv[s][rb].y : kZeroWord,
                                    inside ? wv[s][rb].z : kZeroWord, inside ? wv[s][rb].w : kZeroWord};
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                int t[4];
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const uint32_t addr = __builtin_amdgcn_perm(dw[m], lane_off, 0x0c0c0000u | ((4u + b) << 8));
                    t[b] = static_cast<int>(*reinterpret_cast<const uint32_t*>(tabb + addr));
                }
                A[rb][m] = v4i{t[0], t[1], t[2], t[3]};
            }
            A[rb][4] = v4i{static_cast<int>(t4_bytes(dw[0])), static_cast<int>(t4_bytes(dw[1])),
                           static_cast<int>(t4_bytes(dw[2])), static_cast<int>(t4_bytes(dw[3]))};
        }
#pragma unroll
        for (int kb = 0; kb < 5; ++kb) {
#pragma unroll
            for (int g = 0; g < T; ++g) {
                const uint4 b = bs[((s * 5u + kb) * T + g) * 64u + lane];
                const v4i B = v4i{static_cast<int>(b.x), static_cast<int>(b.y), static_cast<int>(b.z), static_cast<int>(b.w)};
#pragma unroll
                for (int rb = 0; rb < 2; ++rb)
                    acc[rb][g] = TOKENS ? __builtin_amdgcn_mfma_i32_32x32x32_i8(A[rb][kb], B, acc[rb][g], 0, 0, 0)
                                        : __builtin_amdgcn_mfma_i32_32x32x32_i8(B, A[rb][kb], acc[rb][g], 0, 0, 0);
            }
        }
    }
    if constexpr (TOKENS) {
        // Lane l holds token l % 32 of the group and, in register r, row 8 (r / 4) + 4 (l / 32) + r % 4 of block rb: a slice's
        // sums go out as 16-byte pieces.
#pragma unroll
        for (int g = 0; g < T; ++g) {
            const uint32_t m = 32u * g + (lane & 31u);
            if (m >= a.M) continue;
            int32_t* out = a.part + (static_cast<size_t>(kz) * a.M + m) * a.rows_p + sb.row0 + lt * 64u + 4u * half;
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4)
                    *reinterpret_cast<int4*>(out + rb * 32 + 8 * r4) =
                        make_int4(acc[rb][g][4 * r4], acc[rb][g][4 * r4 + 1], acc[rb][g][4 * r4 + 2], acc[rb][g][4 * r4 + 3]);
        }
        return;
    }
    // The product is transposed as gemm_kernel's: lane l holds row l % 32 of block rb and, in register r, token 8 (r / 4) +
    // 4 (l / 32) + r % 4, so that a store writes 128 consecutive bytes of two tokens.
    int32_t* out = a.kslices == 1 ? sb.y : a.part + static_cast<size_t>(kz) * a.M * a.rows_p + sb.row0;
    const uint32_t ld = a.kslices == 1 ? sb.ldy : a.rows_p;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
        const uint32_t n = lt * 64u + rb * 32u + (lane & 31u);
        if (a.kslices == 1 && n >= sb.rows) continue;
#pragma unroll
        for (int r4 = 0; r4 < 4 * T; ++r4) {
            if (8u * r4 >= a.M) break;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t m = 8u * r4 + 4u * half + e;
                if (m < a.M) out[static_cast<size_t>(m) * ld + n] = acc[rb][r4 / 4][4 * (r4 % 4) + e];
            }
        }
    }
}

// The small kernel's shape for T token groups: waves per workgroup (4 or 8) and K steps per slice (2 to kSmallSteps). A
// round is one workgroup per CU (the trit table and the B fragments take 104-144 KiB of LDS); a round costs about 3 K
// steps of loads and staging plus its K steps, each T W / 4 one-wave steps of matrix-core work per SIMD, and the finish
// about a quarter step per slice (measured at 23040 x 3072 and 3072 x 23040). The cheapest pair; on a tie the longer slices.
struct SmallShape {
    uint32_t waves, steps, kslices;
};

static SmallShape small_shape(const Geometry& g, int num_cus, uint32_t T) {
    const uint32_t n_ksteps = static_cast<uint32_t>((g.n_chunks + kStepChunks - 1) / kStepChunks);
    const uint32_t n_tiles = static_cast<uint32_t>(g.n_tiles), cus = static_cast<uint32_t>(std::max(num_cus, 1));
    double best = 1e300;
    SmallShape sh{4, kSmallSteps, 1};
    for (uint32_t st = kSmallSteps; st >= 2; --st) {
        const uint32_t ks = (n_ksteps + st - 1) / st;
        for (uint32_t w : {4u, 8u}) {
            const uint32_t rounds = ((n_tiles + w - 1) / w * ks + cus - 1) / cus;
            const double cost = static_cast<double>(rounds) * (3.0 + st * T * w / 4.0) + (ks > 1 ? 0.25 * ks : 0.0);
            if (cost < best - 1e-9) {
                best = cost;
                sh = SmallShape{w, st, ks};
            }
        }
    }
    return sh;
}

// ---- host side ---------------------------------------------------------------------------------------------------------

// The call's matrices concatenated (tiles, and rows of the slice sums).
static Geometry group_geometry(const GemmSub* subs, int n) {
    size_t rows_p = 0;
    for (int i = 0; i < n; ++i) rows_p += subs[i].g->padded_rows;
    return geometry(rows_p, subs[0].g->cols);
}

static uint32_t token_groups(size_t M) { return static_cast<uint32_t>((M + 31) / 32); }

size_t gemm_ksteps(size_t cols) { return (geometry(1, cols).n_chunks + kStepChunks - 1) / kStepChunks; }

size_t gemm_stage_bytes(size_t cols, size_t M) {
    return M <= kGemmSmallM ? 0 : round_up(gemm_ksteps(cols) * 5u * token_groups(M) * 1024u, 256);
}

struct GemmPlan {
    uint32_t T, R, n_tt, n_rg, kslices, steps;
};

// The tile (T token groups, R blocks per wave) and the K slices of least estimated time, in us: 7 for the call and, per
// K step, 0.4 + 0.095 T R for a workgroup alone on a CU (0.068 T R of it matrix work at 2.4 GHz; a wave issues an
// instruction every 7 cycles or so, which keeps the rest from running beside it), 0.7 of that for each of several on
// one CU, plus for more than one slice the finish kernel, 3.5 and its traffic. Over 337 products of 64 x 4096 to 46080 x
// 3072 and 33 to 1500 tokens, each timed with every tile and up to 19 numbers of slices, the choice was 1.8 % slower than
// the best on average, more than 10 % in 12 of them. Slice sums are kept within the scratch of the no-allocation entry point.
static GemmPlan gemm_plan(const Geometry& g, size_t M, int num_cus) {
    const uint32_t n_ksteps = static_cast<uint32_t>(gemm_ksteps(g.cols));
    const uint32_t n_tg = token_groups(M);
    const uint64_t blocks = 2 * g.n_tiles, cus = static_cast<uint64_t>(std::max(num_cus, 1));
    const size_t xs = gemm_stage_bytes(g.cols, M), out = M * g.padded_rows * 4u;
    GemmPlan best{};
    double best_t = 1e300;
    constexpr uint32_t kShapes[][2] = {{4, 3}, {4, 1}, {2, 2}, {2, 1}};
    for (const auto& sh : kShapes) {
        const uint32_t T = sh[0], R = sh[1];
        if (T > 2 && n_tg <= 2) continue;
        GemmPlan p{T, R, (n_tg + T - 1) / T, static_cast<uint32_t>((blocks + 4 * R - 1) / (4 * R)), 1, n_ksteps};
        const double step = 0.4 + 0.095 * T * R;
        for (uint32_t want = 1; want <= std::min<uint32_t>(n_ksteps, 32u); ++want) {
            p.steps = (n_ksteps + want - 1) / want;
            p.kslices = (n_ksteps + p.steps - 1) / p.steps;
            if (p.kslices != want) continue;
            if (want > 1 && xs + want * out > kNoAllocScratchBytes) break;
            const uint64_t per_cu = (static_cast<uint64_t>(p.n_rg) * p.n_tt * want + cus - 1) / cus;
            double t = 7.0 + p.steps * step * per_cu * (per_cu > 1 && T * R < 8 ? 0.7 : 1.0);
            if (want > 1) t += 3.5 + 2.0 * want * out * 0.2e-6;
            if (t < best_t) {
                best_t = t;
                best = p;
            }
        }
    }
    return best;
}

// Whether a call on x itself (raw; fragments that the caller has staged take the tiled kernel) of more than 32 tokens takes
// the small kernel with two token groups: in one round of workgroups of long slices, where all of a slice's weights in
// flight beat the tiled kernel's three steps ahead. Small against tiled at 33 and 64 tokens: 3072 x 23040 (7 K steps) 15.9
// against 19.1 and 19.2 against 20.6 us, 8192 x 6912 (6) 12.7 against 14.5 and 15.8 against 18.2, 4000 x 18000 (8) 14.5
// against 17.2 and 17.6 against 19.4 (at worst, 4000 x 16001 x 64, 22.7 against 20.3); with shorter slices 3072 x 14336
// (5) 15.7 against 16.9 and 19.6 against 17.1, 2560 x 9216 (3) 13.1 against 12.1 and 17.1 against 14.3; beyond 128 tiles
// 17132 x 2562 x 63 (6) 25.7 against 15.9.
static bool small_form(const Geometry& g, size_t M, bool raw, int num_cus) {
    if (M <= kGemmSmallM) return true;
    if (!raw || M > 64) return false;  // (raw calls are of one matrix)
    const SmallShape sh = small_shape(g, num_cus, 2u);
    return g.n_tiles <= 128u && sh.waves == 4u && sh.steps >= 6u && sh.kslices > 1u &&
           (g.n_tiles + 3) / 4 * sh.kslices <= static_cast<size_t>(std::max(num_cus, 1));
}

size_t gemm_group_part_bytes(const GemmSub* subs, int n, size_t M, bool raw, int num_cus) {
    const Geometry g = group_geometry(subs, n);
    const uint32_t ks = small_form(g, M, raw, num_cus) ? small_shape(g, num_cus, token_groups(M)).kslices : gemm_plan(g, M, num_cus).kslices;
    return ks > 1 ? round_up(static_cast<size_t>(ks) * M * g.padded_rows * 4u, 256) : 0;
}

size_t gemm_workspace_bytes(const Geometry& g, size_t M, int num_cus) {
    const GemmSub sub{nullptr, &g, nullptr, 0};
    return std::max<size_t>(gemm_stage_bytes(g.cols, M) + gemm_group_part_bytes(&sub, 1, M, true, num_cus), 256);
}

template <bool RAW>
static void launch_tiles(const GemmPlan& p, const GemmArgs& a, hipStream_t stream) {
    const dim3 grid(static_cast<uint32_t>(round_up(p.n_rg * p.kslices * p.n_tt, 8))), block(256);
    if (p.T == 4) {
        if (p.R == 3) hipLaunchKernelGGL((gemm_kernel<4, 3, RAW>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((gemm_kernel<4, 1, RAW>), grid, block, 0, stream, a);
    } else {
        if (p.R == 2) hipLaunchKernelGGL((gemm_kernel<2, 2, RAW>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((gemm_kernel<2, 1, RAW>), grid, block, 0, stream, a);
    }
}

// Slices of more than 16 tokens are stored with the tokens in the lanes (8 stores a wave and token group instead of up to
// 32: 300 x 1600 x 32 7.4 -> 7.1 us, 1024 x 3072 x 32 11.1 -> 10.7); at 8 tokens both take as many, and rows in the lanes
// write whole lines (3072 x 23040 x 8 11.1 -> 10.8).
template <int W>
static void launch_small(const GemmArgs& a, hipStream_t stream) {
    const dim3 grid((a.n_tiles + W - 1) / W, a.kslices), block(W * 64);
    const bool tokens = a.kslices > 1u && a.M > 16u;
    if (a.n_sub > 1u) {
        if (tokens) hipLaunchKernelGGL((gemm_small_kernel<1, W, true, true>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((gemm_small_kernel<1, W, true, false>), grid, block, 0, stream, a);
    } else {
        if (tokens) hipLaunchKernelGGL((gemm_small_kernel<1, W, false, true>), grid, block, 0, stream, a);
        else hipLaunchKernelGGL((gemm_small_kernel<1, W, false, false>), grid, block, 0, stream, a);
    }
}

int launch_gemm_group(const GemmSub* subs, int n, int num_cus, const int8_t* x, size_t M, size_t ldx, uint8_t* staged,
                      uint8_t* part, hipStream_t stream) {
    if (n < 1 || n > kGemmSubs) VX_FAIL(VX_ERR_INTERNAL, "a GEMM of %d matrices", n);
    for (int i = 1; i < n; ++i)
        if (subs[i].g->cols != subs[0].g->cols) VX_FAIL(VX_ERR_INTERNAL, "a grouped GEMM of different columns");
    const Geometry g = group_geometry(subs, n);
    GemmArgs a{};
    a.n_sub = static_cast<uint32_t>(n);
    uint32_t tiles = 0, rows_p = 0;
    for (int i = 0; i < n; ++i) {
        const Geometry& gi = *subs[i].g;
        a.sub[i] = GemmMat{subs[i].w, subs[i].y, static_cast<uint32_t>(subs[i].ldy), static_cast<uint32_t>(gi.rows),
                           static_cast<uint32_t>(gi.padded_rows), static_cast<uint32_t>(gi.n_tiles), tiles, rows_p};
        tiles += static_cast<uint32_t>(gi.n_tiles);
        rows_p += static_cast<uint32_t>(gi.padded_rows);
    }
    a.x = x;
    a.xs = reinterpret_cast<const u32x4g*>(staged);
    a.part = reinterpret_cast<int32_t*>(part);
    a.ldx = static_cast<uint32_t>(ldx);
    a.rows_p = rows_p;
    a.cols = static_cast<uint32_t>(g.cols);
    a.n_tiles = tiles;
    a.n_chunks = static_cast<uint32_t>(g.n_chunks);
    a.n_ksteps = static_cast<uint32_t>((g.n_chunks + kStepChunks - 1) / kStepChunks);
    a.M = static_cast<uint32_t>(M);
    a.n_tg = token_groups(M);
    if (small_form(g, M, x != nullptr, num_cus)) {
        const SmallShape sh = small_shape(g, num_cus, token_groups(M));
        a.kslices = sh.kslices;
        a.steps = sh.steps;
        if (M > kGemmSmallM) {  // small_form: several slices of one matrix, 4 waves
            if (n != 1 || sh.waves != 4u || sh.kslices < 2u) VX_FAIL(VX_ERR_INTERNAL, "a small GEMM of %zu tokens", M);
            hipLaunchKernelGGL((gemm_small_kernel<2, 4, false, true>), dim3((a.n_tiles + 3) / 4, a.kslices), dim3(256), 0, stream, a);
        } else if (sh.waves == 8) launch_small<8>(a, stream);
        else launch_small<4>(a, stream);
    } else {
        const GemmPlan p = gemm_plan(g, M, num_cus);
        a.kslices = p.kslices;
        a.steps = p.steps;
        a.n_rg = p.n_rg;
        a.n_tt = p.n_tt;
        if (x == nullptr) {  // staged by the caller
            launch_tiles<false>(p, a, stream);
        } else if (g.cols % 16 == 0) {
            launch_tiles<true>(p, a, stream);
        } else {
            hipLaunchKernelGGL(gemm_stage_kernel, dim3((2u * a.n_ksteps + kStageRows - 1) / kStageRows, a.n_tg), dim3(256), 0,
                               stream, x, a.ldx, a.n_tg, a.cols, a.n_ksteps, reinterpret_cast<u32x4g*>(staged), a.M);
            VX_HIP(hipGetLastError());
            launch_tiles<false>(p, a, stream);
        }
    }
    VX_HIP(hipGetLastError());
    if (a.kslices > 1) {
        const dim3 grid((a.rows_p + 255u) / 256u, a.M);
        if (n > 1) hipLaunchKernelGGL(gemm_finish_kernel<true>, grid, dim3(256), 0, stream, a);
        else hipLaunchKernelGGL(gemm_finish_kernel<false>, grid, dim3(256), 0, stream, a);
        VX_HIP(hipGetLastError());
    }
    return VX_OK;
}

int launch_gemm(const uint8_t* w, const Geometry& g, int num_cus, const int8_t* x, size_t M, size_t ldx, int32_t* y,
                size_t ldy, uint8_t* ws, hipStream_t stream) {
    const GemmSub sub{w, &g, y, ldy};
    return launch_gemm_group(&sub, 1, num_cus, x, M, ldx, ws, ws + gemm_stage_bytes(g.cols, M), stream);
}

// ---- the no-allocation entry point's workspace -----------------------------------------------------------------------

// Workspace of vx_gemm_i32_noalloc_dev: one array per GPU, allocated with the code object when the library's kernels
// are first loaded on that GPU and held until the process ends. Host code never passes `scratch` itself (in host code
// the name is only a stand-in for the symbol); it passes the device address hipGetSymbolAddress returns for the
// current device, looked up once per device. Every call on a GPU reuses that GPU's array, so calls that overlap on one
// GPU race. The kernels write every word of the K-slice sums that they later read; stale fragments of tokens past M are
// read too, but reach only outputs that are never stored. So no clearing is needed between calls.
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

constexpr int kMaxScratchDevices = 64;
static std::mutex g_scratch_mu;
static uint8_t* g_scratch_ptr[kMaxScratchDevices] = {};

// The device address of `scratch` on `device`, which must be the current device.
static int scratch_address(int device, uint8_t** out) {
    if (device < 0 || device >= kMaxScratchDevices)
        VX_FAIL(VX_ERR_UNSUPPORTED, "device %d is beyond the %d devices the no-allocation GEMM serves", device,
                kMaxScratchDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device] == nullptr) {
        void* p = nullptr;
        VX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (p == nullptr) VX_FAIL(VX_ERR_DEVICE, "hipGetSymbolAddress returned no address for the GEMM scratch");
        g_scratch_ptr[device] = static_cast<uint8_t*>(p);
    }
    *out = g_scratch_ptr[device];
    return VX_OK;
}

int gemm_scratch_prepare(int device) {
    uint8_t* p = nullptr;
    return scratch_address(device, &p);
}

int launch_gemm_noalloc(const uint8_t* w, const Geometry& g, int device, int num_cus, const int8_t* x, size_t M,
                        size_t ldx, int32_t* y, size_t ldy, hipStream_t stream) {
    const size_t need = gemm_workspace_bytes(g, M, num_cus);
    if (need > kNoAllocScratchBytes)
        VX_FAIL(VX_ERR_INVALID_SHAPE,
                "m = %zu tokens on a %zu x %zu matrix need %zu bytes of workspace, more than the %zu bytes the "
                "no-allocation GEMM holds; use vx_gemm_i32_dev with a workspace",
                M, g.rows, g.cols, need, kNoAllocScratchBytes);
    uint8_t* ws = nullptr;
    VX_TRY(scratch_address(device, &ws));
    return launch_gemm(w, g, num_cus, x, M, ldx, y, ldy, ws, stream);
}

}  // namespace vx
