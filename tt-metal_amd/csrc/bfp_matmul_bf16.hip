// GEMM with two bf16 operands for gfx950, the weights read where they lie: 4-face tiles, no pass that lays them out first.
//
// What it is for: batched products whose operands are both activations (scores and context of an attention layer: every
// head brings weights of its own, used once), where a re-layout pass costs as much as the product, and outputs too small
// or too narrow for the 256 x 256 blocks of matmul_expanded_kernel.  Those products move more bytes than they have work
// for the matrix cores (8 x 16 heads of [384, 64] x [64, 384]: 50 MB, 2.4 GFLOP), so HBM bounds them.  Block-float weights come
// here, expanded to bf16 tiles by expand_tiles_kernel, where blocks of 64 or 128 fill the chip and 256 x 256 ones do not.
//
//   block      32 RB WR rows x 32 CB WC columns of C per workgroup of four wavefronts (WR x WC of them)
//   staging    one k tile row (32 k values) per step, whole tiles of A and B through a ring of LDS stages filled by direct
//              global->LDS loads; a lane may fetch any 16 bytes, so the swizzles below cost nothing
//   A          chunk (row r, half h) of a face lies at r * 32 + (h ^ (r / 8)) * 16: the 16 lanes of one pass of a
//              ds_read_b128 find 16 different bank groups (without the XOR rows r and r + 8 share theirs)
//   B          a lane needs 8 consecutive k rows of one column, and a tile holds rows: ds_read_b64_tr_b16 transposes on
//              the way.  Sixteen lanes read 4 rows x 16 columns (128 contiguous bytes), lane l gets column l.  The two
//              128-byte halves of the row groups are exchanged in the right-hand faces, so that the two 16-lane groups
//              of one pass (faces 2s and 2s + 1) lie in different halves of the 64 banks
//   math       v_mfma_f32_32x32x16_bf16 with B's columns as the rows of the product: accumulator element i of lane
//              (c = lane % 32, kh = lane / 32) is row c of the 32 rows and column 8 (i / 4) + 4 kh + i % 4.  Four adjacent
//              columns per lane; v_permlane32_swap joins them to eight, and C is stored with 16 bytes per lane straight
//              from registers, whole face rows, with no staging
// Semantics as in bfp_matmul.hip (tt::operations::primary::matmul, tt_eager/tt_dnn/op_library/bmm/bmm_op.hpp:318-346).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "bfp_dequant.h"
#include "ttmi_internal.h"

namespace ttmi {

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

struct DirectDev {
    const uint8_t *a;        // bf16
    const uint8_t *b;        // bf16 tiles
    const uint16_t *bias;    // bf16, n columns (bias_at), or null
    uint8_t *c;
    uint32_t b_batch, m, k, n;
    uint32_t kt, nt, mt, tiles_m, tiles_n, blocks, per_xcd;
    int a_tiled, c_tiled, c_f32, bias_tiled;
    int c_bfp;               // 0, or the mantissa bits (7 | 3) of a block-float output in TILE layout
    float unscale;           // common factor of the products: 1, or Wfmt::unscale for expanded block floats
};

// LDS reads are written as inline assembly: the compiler orders every transposing read behind ALL outstanding direct-to-LDS
// loads (it cannot tell that they write other stages), which would drain the ring at every step.  The waits carry the
// results as operands, so that nothing that uses them can be scheduled in front.
__device__ __forceinline__ void read_transposed(u32x2 &v, uint32_t at, int offset) {
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(offset));
}
// slab 0: all but the reads of slab 1 (issued last) have returned; slab 1: all
template <int RB, int CB> __device__ __forceinline__ void wait_operands(u32x4 (&a)[RB], u32x2 (&b)[CB][2], int s) {
    constexpr int younger = RB + 2 * CB;
    if (s == 0) asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(younger) : "memory");
    else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < RB; ++i) asm volatile("" : "+v"(a[i]));
#pragma unroll
    for (int i = 0; i < CB; ++i) asm volatile("" : "+v"(b[i][0]), "+v"(b[i][1]));
}

template <int ACT, int WR, int WC, int RB, int CB, int STAGES>
__global__ __launch_bounds__(256, 2) void matmul_direct_kernel(const DirectDev p) {
    static_assert(WR * WC == 4, "four wavefronts");
    constexpr int BANDS = WR * RB, COLS = WC * CB;              // 32-row bands and 32-column tiles of a block
    constexpr int STAGE_BYTES = (BANDS + COLS) * 2048;
    constexpr int LOADS = (BANDS + COLS) * 2 / 4;               // 1 KiB each, per wavefront and step
    static_assert((BANDS + COLS) % 2 == 0 && STAGES >= 3, "every wavefront requests the same number of pieces");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[STAGES * STAGE_BYTES];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave / WC, wc = wave % WC;
    const int c = lane & 31, kh = lane >> 5;

    // consecutive workgroups go to the 8 XCDs in turn: each XCD takes a contiguous run of blocks, so that the blocks of a
    // slice share one L2's copy of its operands
    const uint32_t block = (blockIdx.x & 7) * p.per_xcd + (blockIdx.x >> 3);
    if (block >= p.blocks) return;                              // the whole workgroup, before any barrier
    uint32_t idx = block;
    const uint32_t tn = idx % p.tiles_n; idx /= p.tiles_n;
    const uint32_t tm = idx % p.tiles_m;
    const uint32_t bb = idx / p.tiles_m;
    const uint32_t band0 = tm * BANDS, nt0 = tn * COLS;

    // ---- requests: piece i of this wavefront is half a tile, 16 bytes per lane --------------------------------------------
    const uint8_t *src[LOADS];
    uint64_t step[LOADS];                                       // a k tile row of B has more than 4 GiB from 2^26 columns on
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const uint32_t piece = wave * LOADS + i, tile = piece >> 1, at = (piece & 1) * 64 + lane;   // 16-byte place in the tile
        const uint32_t face = at >> 5, within = at & 31;
        if (tile < (uint32_t)BANDS) {
            const uint32_t r = within >> 1, h = (within & 1) ^ (r >> 3);
            const uint32_t band = min(band0 + tile, p.mt - 1);                                      // past the last band: any valid memory
            if (p.a_tiled) {
                src[i] = p.a + ((uint64_t)bb * p.mt + band) * p.kt * 2048 + face * 512 + r * 32 + h * 16;
                step[i] = 2048;
            } else {
                const uint32_t row = min(band * 32 + (face >> 1) * 16 + r, p.m - 1);
                src[i] = p.a + ((uint64_t)bb * p.m + row) * p.k * 2 + (face & 1) * 32 + h * 16;
                step[i] = 64;
            }
        } else {
            const uint32_t col = min(nt0 + tile - BANDS, p.nt - 1);
            src[i] = p.b + ((uint64_t)(p.b_batch == 1 ? 0 : bb) * p.kt * p.nt + col) * 2048 + face * 512 + (within ^ ((face & 1) * 8)) * 16;
            step[i] = (uint64_t)p.nt * 2048;
        }
    }
    auto request = [&](uint32_t stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src[i],
                                             (__attribute__((address_space(3))) void *)(lds + stage * STAGE_BYTES + (wave * LOADS + i) * 1024), 16, 0, 0);
            src[i] += step[i];
        }
    };

    const uint32_t lds_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    const uint32_t a_at = (wr * RB) * 2048 + (c >> 4) * 1024 + (c & 15) * 32 + ((kh ^ ((c >> 3) & 1)) * 16);      // + slab * 512
    const uint32_t fc = (lane >> 4) & 1, l16 = lane & 15;
    const uint32_t b_at = (BANDS + wc * CB) * 2048 + fc * 512 + kh * 256 + fc * 128 + l16 * 8;                   // + slab * 1024; the other half: ^ 128

    f32x16 acc[RB][CB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[rb][cb][r] = 0.f;

    uint32_t asked = 0;
    for (; asked < STAGES - 1 && asked < p.kt; ++asked) request(asked);
    uint32_t stage = 0, ask_stage = STAGES - 1;
#pragma unroll 1
    for (uint32_t t = 0; t < p.kt; ++t) {
        // step t has landed for everybody, and nobody reads the stage of step t - 1 any more
        if (asked - t == STAGES - 1) wait_vmcnt<(STAGES - 2) * LOADS>();
        else wait_vmcnt<0>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (asked < p.kt) { request(ask_stage); ++asked; }
        const uint32_t from = lds_at + stage * STAGE_BYTES;
        // both slabs' operands are requested at once; the second slab's arrive under the first one's MFMAs
        u32x4 a[2][RB];
        u32x2 b[2][CB][2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                read_transposed(b[s][cb][0], from + b_at, cb * 2048 + s * 1024);
                read_transposed(b[s][cb][1], from + (b_at ^ 128u), cb * 2048 + s * 1024);
            }
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(a[s][rb]) : "v"(from + a_at), "n"(rb * 2048 + s * 512));
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            wait_operands<RB, CB>(a[s], b[s], s);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) {
                    const u32x4 w = u32x4{b[s][cb][0][0], b[s][cb][0][1], b[s][cb][1][0], b[s][cb][1][1]};
                    acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a[s][rb]), acc[rb][cb], 0, 0, 0);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        ask_stage = ask_stage + 1 == STAGES ? 0 : ask_stage + 1;
    }

    // ---- store --------------------------------------------------------------------------------------------------------------
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const uint32_t band = band0 + wr * RB + rb, row = band * 32 + c;
        if (band >= p.mt) break;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const uint32_t col_tile = nt0 + wc * CB + cb;
            if (col_tile >= p.nt) break;
            const uint64_t tile = ((uint64_t)bb * p.mt + band) * p.nt + col_tile;
#pragma unroll
            for (int f = 0; f < 2; ++f) {                       // the columns of one face: accumulator quads 2f and 2f + 1
                float v[8];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    uint2 bias4 = make_uint2(0u, 0u);
                    if (p.bias) __builtin_memcpy(&bias4, p.bias + bias_at(col_tile * 32 + f * 16 + h * 8 + kh * 4, p.bias_tiled), 8);      // a bias need not be aligned
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t w = i < 2 ? bias4.x : bias4.y;
                        v[h * 4 + i] = apply_activation<ACT>(acc[rb][cb][(2 * f + h) * 4 + i] * p.unscale + __uint_as_float((i & 1) ? w & 0xffff0000u : w << 16));
                    }
                }
                if (p.c_f32) {
                    if (row < p.m) {
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            const uint32_t col = h * 8 + kh * 4;
                            const uint64_t elem = p.c_tiled ? tile * 1024 + ((c >> 4) * 2 + f) * 256 + (c & 15) * 16 + col
                                                            : ((uint64_t)bb * p.m + row) * p.n + col_tile * 32 + f * 16 + col;
                            *reinterpret_cast<float4 *>(p.c + elem * 4) = make_float4(v[h * 4], v[h * 4 + 1], v[h * 4 + 2], v[h * 4 + 3]);
                        }
                    }
                    continue;
                }
                // columns 0-3 | 4-7 of quad 2f and 8-11 | 12-15 of quad 2f + 1 sit in the lanes kh = 0 | 1: the swap leaves
                // columns 8 kh .. 8 kh + 7 of the face row in each lane
                const auto w0 = __builtin_amdgcn_permlane32_swap(f32x2_to_bf16x2_rne(v[0], v[1]), f32x2_to_bf16x2_rne(v[4], v[5]), false, false);
                const auto w1 = __builtin_amdgcn_permlane32_swap(f32x2_to_bf16x2_rne(v[2], v[3]), f32x2_to_bf16x2_rne(v[6], v[7]), false, false);
                const u32x4 out = u32x4{w0[0], w1[0], w0[1], w1[1]};
                if (p.c_bfp) {
                    // the host packers' arithmetic on the bf16-rounded sums; a face row is the two lanes c and c + 32
                    uint32_t bits[8], shared = 0;
#pragma unroll
                    for (int i = 0; i < 4; ++i) { bits[2 * i] = out[i] << 16; bits[2 * i + 1] = out[i] & 0xffff0000u; }
#pragma unroll
                    for (int i = 0; i < 8; ++i) shared = max(shared, (bits[i] >> 23) & 0xffu);
                    const auto other = __builtin_amdgcn_permlane32_swap(shared, shared, false, false);
                    shared = max(other[0], other[1]);
                    const uint32_t face = (c >> 4) * 2 + f, r16 = c & 15;
                    uint8_t *to = p.c + tile * (p.c_bfp == 7 ? 1088u : 576u);
                    if (p.c_bfp == 7) {
                        uint32_t words[2] = {0, 0};
#pragma unroll
                        for (int i = 0; i < 8; ++i) words[i >> 2] |= to_code<7>(bits[i], shared) << (8 * (i & 3));
                        *reinterpret_cast<uint2 *>(to + 64 + face * 256 + r16 * 16 + kh * 8) = make_uint2(words[0], words[1]);
                    } else {
                        uint32_t word = 0;
#pragma unroll
                        for (int i = 0; i < 8; ++i) word |= to_code<3>(bits[i], shared) << (4 * i);
                        *reinterpret_cast<uint32_t *>(to + 64 + face * 128 + r16 * 8 + kh * 4) = word;
                    }
                    if (kh == 0) to[face * 16 + r16] = (uint8_t)shared;
                } else if (p.c_tiled) {
                    *reinterpret_cast<u32x4 *>(p.c + tile * 2048 + ((c >> 4) * 2 + f) * 512 + (c & 15) * 32 + kh * 16) = out;
                } else if (row < p.m) {
                    *reinterpret_cast<u32x4 *>(p.c + (((uint64_t)bb * p.m + row) * p.n + col_tile * 32 + f * 16 + kh * 8) * 2) = out;
                }
            }
        }
    }
}

// Packed tiles -> bf16 tiles in the same element order, for a GEMM of block-float weights on the kernel above: 8 elements per lane
// and piece, four pieces in flight.  HBM-bound.  The values carry the common factor of Wfmt::unscale, and the ends of the
// exponent range come out as in expand_kernel.
template <int W>
__global__ __launch_bounds__(256) void expand_tiles_kernel(const uint8_t *__restrict__ b, u32x4 *__restrict__ out, uint64_t pieces) {
    constexpr int PIECES = 4;
    const uint64_t first = (uint64_t)blockIdx.x * (256 * PIECES) + threadIdx.x;
    uint32_t words[PIECES][2], exps[PIECES];
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
        const uint64_t at = min(first + j * 256, pieces - 1);
        const uint32_t piece = (uint32_t)at & 127;                       // of the tile's 128
        const uint8_t *tile = b + (at >> 7) * Wfmt<W>::tile_bytes;
        exps[j] = tile[piece >> 1];
        if (W == 7) {
            const uint2 v = *reinterpret_cast<const uint2 *>(tile + 64 + piece * 8);
            words[j][0] = v.x; words[j][1] = v.y;
        } else {
            words[j][0] = *reinterpret_cast<const uint32_t *>(tile + 64 + piece * 4);
        }
    }
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
        const float scale = row_scale(exps[j]);
        u32x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t bits[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int e = 2 * i + h;
                const uint32_t code = W == 7 ? words[j][e >> 2] >> (8 * (e & 3)) : words[j][0] >> (4 * e);
                bits[h] = __float_as_uint((float)(code & ((1u << W) - 1)) * scale) | ((code >> W) & 1u) << 31;      // at most 7 significant bits
            }
            v[i] = (bits[1] & 0xffff0000u) | bits[0] >> 16;
        }
        if (first + j * 256 < pieces) out[first + j * 256] = v;
    }
}

namespace {
template <int WR, int WC, int RB, int CB, int STAGES> int launch_direct(DirectDev p, const MatmulArgs &x, hipStream_t st) {
    p.tiles_m = (p.mt + WR * RB - 1) / (WR * RB);
    p.tiles_n = (p.nt + WC * CB - 1) / (WC * CB);
    const uint64_t blocks = (uint64_t)x.batch * p.tiles_m * p.tiles_n;
    if (blocks > 0x7ffffff0ull) return fail(TTMI_ERR_INVALID_ARGUMENT, "matmul: problem too large for one launch");
    p.blocks = (uint32_t)blocks;
    p.per_xcd = (p.blocks + 7) / 8;
    const dim3 grid(p.per_xcd * 8);
    switch (x.activation) {
        case TTMI_ACT_RELU: hipLaunchKernelGGL((matmul_direct_kernel<TTMI_ACT_RELU, WR, WC, RB, CB, STAGES>), grid, dim3(256), 0, st, p); break;
        case TTMI_ACT_GELU: hipLaunchKernelGGL((matmul_direct_kernel<TTMI_ACT_GELU, WR, WC, RB, CB, STAGES>), grid, dim3(256), 0, st, p); break;
        case TTMI_ACT_SILU: hipLaunchKernelGGL((matmul_direct_kernel<TTMI_ACT_SILU, WR, WC, RB, CB, STAGES>), grid, dim3(256), 0, st, p); break;
        default: hipLaunchKernelGGL((matmul_direct_kernel<TTMI_ACT_NONE, WR, WC, RB, CB, STAGES>), grid, dim3(256), 0, st, p); break;
    }
    return check_launch("matmul_direct_kernel");
}
}  // namespace

// Rows and columns of the block a shape goes to, 0 for the re-layout and 256 x 256 blocks.  Estimates from these
// measurements (us, one MI355X; 64 / 128 / 256 blocks): a k tile row takes a 128 x 128 block 0.31 us alone on its CU and 0.27
// as one of several ([512, 2048] x [2048, 2048], a quarter of the chip: 22 us; [2048, 4096] x [4096, 4096], two per CU: 68); a
// 64 x 64 block 0.165 us alone and 0.143 us as one of many, 0.1 where the weights are few columns, which every L2 keeps
// ([256, 8192] x [8192, 1024] 43 / 74 / 144, [4096, 4096] x [4096, 4096] 293 / 159 / 130, [3072, 4096] x [4096, 1024], block-float
// weights, 44 / 47 / 53); a 256 x 256 block 0.72 us behind a pass over the weights and a second launch.
// What the line at 1024 columns stands for is a jump of 64 blocks there, 128 ones do not have it.  BFLOAT8_B weights, the pass
// over them included, 64 / 128 blocks at n = 768, 992, 1024, 1056, 1280, 1536, 2048:
//   [2048, 4096] x [4096, n]  35/46 36/46 37/46 48/47 54/48 58/49 82/51
//   [1024, 4096] x [4096, n]  31/47 32/47 30/46 34/47 34/47 37/48 40/49
//   [3072, 4096] x [4096, n]  49/46 53/47 54/47 65/48 72/49 87/69 118/71
//   [3072, 1024] x [1024, n]  17/18 19/19 20/19 22/20 23/21 27/25 33/26
// so 0.1 is too little at 3072 rows (12 % lost up to 1024 columns on that box), and the estimate of 128 blocks too much from 1056 on.
static double direct_us(uint32_t batch, uint32_t m, uint32_t k, uint32_t n, uint32_t *block) {
    const double steps = k / 32;
    auto blocks = [&](uint32_t edge) { return (double)batch * ((m + edge - 1) / edge) * ((n + edge - 1) / edge) / 256.0; };
    const double at64 = steps * std::max(0.165, blocks(64) * (n <= 1024 ? 0.1 : 0.143)),
                 at128 = steps * (blocks(128) <= 1.0 ? 0.31 : std::ceil(blocks(128)) * 0.27);
    if (block) *block = at64 < at128 ? 64 : 128;
    return std::min(at64, at128);
}
uint32_t bf16_direct_block(uint32_t batch, uint32_t b_batch, uint32_t m, uint32_t k, uint32_t n) {
    uint32_t block;
    const double direct = direct_us(batch, m, k, n, &block), blocks = (double)batch * ((m + 255) / 256) * ((n + 255) / 256);
    return 8.0 + (double)b_batch * k * n * 4.0 / 5.0e6 + (k / 32) * std::ceil(blocks / 256.0) * 0.72 < direct ? 0 : block;
}
// With a pass in front that expands block-float weights to bf16 tiles.
double matmul_direct_estimate(uint32_t batch, uint32_t b_batch, uint32_t m, uint32_t k, uint32_t n, double bytes_per_weight) {
    return 5.0 + (double)b_batch * k * n * (bytes_per_weight + 2.0) / 4.0e6 + direct_us(batch, m, k, n, nullptr);
}

size_t matmul_direct_scratch_bytes(uint32_t b_batch, uint32_t k, uint32_t n) { return (size_t)b_batch * (k / 32) * (n / 32) * 2048; }

int matmul_bf16_direct(const MatmulArgs &x, hipStream_t st) {
    DirectDev p{};
    p.a = (const uint8_t *)x.a; p.b = (const uint8_t *)x.b; p.bias = (const uint16_t *)x.bias; p.bias_tiled = x.bias_tiled; p.c = (uint8_t *)x.c;
    p.b_batch = x.b_batch; p.m = x.m; p.k = x.k; p.n = x.n;
    p.kt = x.k / 32; p.nt = x.n / 32; p.mt = (x.m + 31) / 32;
    p.a_tiled = x.a_layout == TTMI_TILE; p.c_tiled = x.c_layout == TTMI_TILE; p.c_f32 = x.c_dtype == TTMI_FLOAT32;
    p.c_bfp = x.c_dtype == TTMI_BFLOAT8_B ? 7 : x.c_dtype == TTMI_BFLOAT4_B ? 3 : 0;
    p.unscale = 1.0f;
    std::unique_lock<std::mutex> launches(expanded_scratch_guard(), std::defer_lock);
    if (x.b_fmt != TTMI_BFLOAT16) {                             // scratch of the library's own, which callers without it do not come here for
        const uint64_t pieces = (uint64_t)x.b_batch * p.kt * p.nt * 128, blocks = (pieces + 1023) / 1024;
        if (blocks > 0x7fffffffull) return fail(TTMI_ERR_INVALID_ARGUMENT, "matmul: problem too large for one launch");
        void *dense;
        bool fresh;
        launches.lock();
        if (int rc = scratch_get(SCRATCH_EXPANDED, st, matmul_direct_scratch_bytes(x.b_batch, x.k, x.n), &dense, &fresh)) return rc;
        if (x.b_fmt == TTMI_BFLOAT8_B)
            hipLaunchKernelGGL((expand_tiles_kernel<7>), dim3((uint32_t)blocks), dim3(256), 0, st, p.b, (u32x4 *)dense, pieces);
        else
            hipLaunchKernelGGL((expand_tiles_kernel<3>), dim3((uint32_t)blocks), dim3(256), 0, st, p.b, (u32x4 *)dense, pieces);
        if (int rc = check_launch("expand_tiles_kernel")) return rc;
        p.b = (const uint8_t *)dense;
        p.unscale = x.b_fmt == TTMI_BFLOAT8_B ? Wfmt<7>::unscale : Wfmt<3>::unscale;
    }
    uint32_t block;
    direct_us(x.batch, x.m, x.k, x.n, &block);
    block = knob_or(TTMI_KNOB_MATMUL_BLOCK, block);
    return block == 128 ? launch_direct<2, 2, 2, 2, 3>(p, x, st) : launch_direct<2, 2, 1, 1, 4>(p, x, st);
}

}  // namespace ttmi
