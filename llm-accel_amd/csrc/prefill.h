// prefill.h -- launch interface of the layer-major prompt path (internal).
//
// The request loop's prompt blocks through whole layers at once: every
// projection is one matrix product over up to kPfMaxRows prompt rows instead
// of one weight stream per 8-row block, and the attention walks the same
// 64-position tiles as the block kernels, so every row's values are those of
// its block.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"

namespace llm {

// Activations as byte planes in the matrix cores' operand order ("xp"):
// x = 256 c + d + 128 with c = x >> 8 and d = (x & 255) - 128, both int8.
// Piece (mt, kc) of 2048 bytes holds rows 32 mt .. + 31 and inputs 32 kc ..
// + 31: 1024 bytes of c, then 1024 of d; lane l, byte b of a plane is row
// 32 mt + l % 32, input 32 kc + 16 (l / 32) + b.  Inputs past the matrix's
// width are x = 0 (c = 0, d = -128).
constexpr size_t pf_xp_bytes(uint32_t rows_pad, uint32_t k_pad) {
    return (size_t)rows_pad * k_pad * 2;
}
// Rows of int16 in the products' own result order ("frag16"): piece (mt,
// nt) of 32 rows x 32 columns is [64 lanes][16], lane l's element 4 j + t
// being row 32 mt + l % 32, column 32 nt + 8 j + 4 (l / 32) + t.
__host__ __device__ constexpr size_t pf_frag16(uint32_t m, uint32_t n, uint32_t nt_count) {
    return (((size_t)(m / 32) * nt_count + n / 32) * 64 + m % 32 + 32 * ((n >> 2) & 1)) * 16 +
           4 * ((n % 32) >> 3) + (n & 3);
}
constexpr uint32_t kPfRowPad = 128;  // rows of every buffer are padded to this

struct PfGemmArgs {
    const int8_t* x;       // xp planes of the rows, K_pad = 128 steps wide
    uint32_t m;            // rows (buffers hold them padded to kPfRowPad)
    uint32_t steps;        // K_pad / 128
    uint32_t n;            // outputs per matrix
    // 12-bit copies (p12, see kernels.h; p1 with EPI_SILU), or the byte
    // planes of matrices held in 16 bits
    const uint8_t *p0, *p1;
    const int8_t *mf0, *mf1;
    uint32_t kq;           // K chunks of 64 that the byte planes / sums cover
    const int32_t *ms0, *ms1;        // per output (sum w >> 8, sum (w & 255) - 128)
    const uint32_t *corr0, *corr1;   // corrections of the 12-bit copies, or null
    const int32_t* rowsum; // sum of each row's inputs (byte planes only)
    int16_t* out;          // frag16 (EPI_STORE; EPI_RESID: the residual sum)
    const int16_t* res;    // frag16 residual (EPI_RESID)
    int8_t* xp_out;        // xp planes: silu(gate) up (EPI_SILU), or the
                           // constant-gain RMSNorm of the sum (EPI_RESID, may be null)
    const int16_t* norm_gamma;
    int32_t norm_gain;
    const uint32_t* silu8; // see ProjArgs
    // split of K over workgroups (chosen by the launcher): the parts' exact
    // sums, and an arrival counter per tile (zero between launches)
    uint32_t parts;
    int64_t* part;
    uint32_t* count;
    size_t part_bytes;
    uint32_t max_tiles;
};
// A launch's shape: 32-row pieces per workgroup, workgroup tiles, parts of K.
struct PfShape {
    uint32_t wm, tiles, parts;
};
PfShape pf_gemm_shape(uint32_t m, uint32_t n, uint32_t steps, int epi);
constexpr size_t pf_part_bytes(const PfShape& s) {
    return (size_t)s.tiles * s.parts * (128 * s.wm * 32) * 8;
}
hipError_t launch_pf_gemm(const PfGemmArgs& a, int epi, hipStream_t st);
// rowsum[r] = sum over k of x[r][k] of xp planes.
hipError_t launch_pf_rowsum(const int8_t* x, uint32_t m, uint32_t steps, int32_t* rowsum,
                            hipStream_t st);

// Row-major rows [m][cols] -> frag16 rows and xp planes of their
// constant-gain RMSNorm (k_pad columns, 0 past cols).
hipError_t launch_pf_init(const int16_t* rows, uint32_t m, uint32_t cols, uint32_t k_pad,
                          const int16_t* gamma, int32_t gain, int16_t* h, int8_t* xp,
                          hipStream_t st);

struct PfAttnArgs {
    const int16_t* qkv;    // frag16 rows q | k | v
    uint32_t qkv_nt;       // its column pieces
    uint32_t m, pos0;      // rows, position of row 0
    const int16_t* rope;   // as AttnArgs
    int16_t *kcache, *vcache;
    uint32_t tiles;        // pages per (layer, KV head)
    uint32_t num_heads, num_kv_heads, group, head_dim;
    int32_t qk_scale;
    const int16_t* exp14;
    // scratch: operand planes of the rotated queries, the K and V pages of
    // [0, pos0 + m), 128 times each K row's sum, and per tile / query block
    // what its rare arithmetic needs
    int8_t *qp, *kp, *vp;
    int32_t* kbias;        // [kv_heads][tiles][64]
    uint32_t* kvflag;      // [2][kv_heads][tiles]: a K / V value saturates
    uint32_t* qflag;       // [heads][rows / 32]: a bank's queries are all -32768
    int8_t* xp_out;        // attention outputs, xp planes of k_pad columns
    uint32_t out_steps;
};
size_t pf_qp_bytes(uint32_t rows_pad, uint32_t heads, uint32_t d);
size_t pf_kp_bytes(uint32_t kv_heads, uint32_t tiles, uint32_t d);
size_t pf_vp_bytes(uint32_t kv_heads, uint32_t tiles, uint32_t d);
// RoPE of the rows' queries and keys, the rows' K / V into the cache, and
// the operand planes of both.
hipError_t launch_pf_kvq(const PfAttnArgs& a, hipStream_t st);
hipError_t launch_pf_attention(const PfAttnArgs& a, hipStream_t st);

// The hidden pairs as the blocks of `block` rows leave them: pair row r
// takes the last of rows [0, m) that a block held as its row r; pair1 the
// FFN output h2, pair0 the attention sublayer's h1 or, for the rows of the
// last block when `final_norm`, the final RMSNorm of h2.
hipError_t launch_pf_finish(const int16_t* h1, const int16_t* h2, uint32_t m, uint32_t cols,
                            uint32_t k_pad, uint32_t block, bool final_norm,
                            const int16_t* gamma, int32_t gain, int16_t* pair0, int16_t* pair1,
                            hipStream_t st);

}  // namespace llm
