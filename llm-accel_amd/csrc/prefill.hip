// prefill.hip -- the layer-major prompt path: prompt rows through whole
// layers as matrix products on the matrix cores (see prefill.h).
#include "prefill.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "attn_common.h"
#include "coherent.h"
#include "fixed_point.h"
#include "kernels.h"
#include "proj_common.h"

namespace llm {
namespace {

typedef int32_t v4i __attribute__((ext_vector_type(4)));
typedef int32_t v16i __attribute__((ext_vector_type(16)));

__device__ __forceinline__ int32_t med3(int32_t v, int32_t lo, int32_t hi) {
    return v < lo ? lo : (v > hi ? hi : v);
}
__device__ __forceinline__ uint32_t pack16(int32_t lo, int32_t hi) {
    return ((uint32_t)lo & 0xffffu) | ((uint32_t)hi << 16);
}
// Byte planes of four int16 values (two packed words): c = x >> 8 and
// d = (x & 255) - 128.
__device__ __forceinline__ uint32_t plane_c(uint32_t w0, uint32_t w1) {
    return __builtin_amdgcn_perm(w1, w0, 0x07050301u);
}
__device__ __forceinline__ uint32_t plane_d(uint32_t w0, uint32_t w1) {
    return __builtin_amdgcn_perm(w1, w0, 0x06040200u) ^ 0x80808080u;
}

// ---------------------------------------------------------------------
// Projection of many rows.  With x = 256 c + d + 128 (xp planes) and
// w = 256 a + b, a and b signed bytes (12-bit weights: b the low byte,
// a in [-8, 8]),
//   sum w x = 65536 sum ac + 256 (sum ad + sum bc) + sum bd + 128 sum w,
// every sum exact in int32 (K <= 16384).  Byte-plane weights (16-bit
// matrices) are w = 256 a + b + 128, which adds 128 sum x.
//
// Wavefronts 2 WM: each 32 rows x 64 output slots (32 outputs of gate and of
// up for EPI_SILU), two over 128 slots, WM over the row pieces; the MFMA's A
// operand is the weights, so a lane's results are runs of 4 outputs of one
// row.  Per 128-input step the weights go through LDS, unpacked once per
// workgroup (double-buffered, one barrier per step, two more steps in
// flight); the activation planes are in operand order and come straight from
// L2, each 32-input piece reloaded for the next step after its last use.
// With four row pieces a workgroup fills a compute unit (two wavefronts per
// SIMD) and takes its items in turn, the next item's loads already under way
// during an item's epilogue.  1,024 rows of config B: gate|up 189 us (369 G
// i8 operations, 2.0 POPS; one item per workgroup 213), Q|K|V 31, O 30, down
// 90 with K in two parts.  A plain loop of these products runs at 3.4 POPS on
// such data (the card's power limit; 4.3 on constant data), so gate|up is
// bounded by 110 us: what is left is the unpacking and epilogue arithmetic
// that shares the SIMDs and the uneven last round (5.4 items per workgroup).
// Measured and not kept: 64 x 64 per wavefront (one per SIMD: 299 us), the
// activations requested two steps ahead (no change), a raised wave priority
// around the products (194 us).  Kernels stay small: with the corrections in
// every variant (40 KB of code) a launch began ~20 us later.
// ---------------------------------------------------------------------
constexpr uint32_t kWHalf = 544, kWPlane = 2 * kWHalf, kWPiece = 2368;  // LDS strides (padded)
constexpr uint32_t kPfItems = 16;  // of a workgroup
constexpr uint32_t kWBuf = 16 * kWPiece;  // [4 n pieces][4 k pieces]
static_assert(kWPiece >= 2 * kWPlane && kWPiece % 16 == 0, "piece holds two planes");

template <typename T>
__device__ __forceinline__ void swap_v(T& a, T& b) {
    const T t = a;
    a = b;
    b = t;
}
// b = the low byte, a = h - 8 + (l >> 7): w + 2048 = 256 h + l.
__device__ __forceinline__ uint32_t p12_signed_high(uint32_t h4, uint32_t l4) {
    const uint32_t t = h4 + ((l4 >> 7) & 0x01010101u);
    return ((t | 0x80808080u) - 0x08080808u) ^ 0x80808080u;
}

// fx_narrow_projection in one rounding: with sum + 8 = 256 t + r, 0 <= r <
// 256, rnd(rnd(sum, 4), 8) = floor((16 t + floor(r / 16) + 128) / 256) =
// floor((t + 8) / 16), and the 32-bit saturation between the two roundings
// lies far outside the 16-bit one.
// 12-bit weights, sum = 65536 ac + 256 x + bd + 128 s: the result saturates
// once |t| passes 2^19, so ac may be clamped to 2^21 in magnitude (256 ac
// then outweighs x and s / 2, at most 2^28.1 and 2^24).
__device__ __forceinline__ int32_t pf_narrow12(int32_t ac, int32_t x, int32_t bd, int32_t sh,
                                               int32_t sl) {
    // sh = s >> 1 plus 8, sl = 128 (s & 1) + 8
    const int32_t t = (med3(ac, -(1 << 21), 1 << 21) << 8) + x + sh + ((bd + sl) >> 8);
    return med3(t >> 4, INT16_MIN, INT16_MAX);
}
__device__ __forceinline__ int32_t pf_narrow64(int64_t sum) {
    const int64_t t = ((sum + 8) >> 8) + 8;
    return t > INT32_MAX ? INT16_MAX
                         : (t < INT32_MIN ? INT16_MIN : med3((int32_t)t >> 4, INT16_MIN, INT16_MAX));
}

template <int WM, int EPI, bool WIDE, bool CORR>
__global__ __launch_bounds__(128 * WM, WM == 4 ? 2 : 1) void pf_gemm_kernel(PfGemmArgs a, uint32_t mtiles,
                                                              uint32_t ntiles) {
    constexpr bool SILU = EPI == EPI_SILU;
    constexpr int NTH = 128 * WM, NP = 1024 / NTH;  // threads, weight pieces per thread
    constexpr uint32_t ITEMS = WM == 4 ? kPfItems : 1;
    __shared__ __attribute__((aligned(16))) uint8_t wl[2 * kWBuf];
    __shared__ int2 sw[ITEMS][128];  // per item a slot's weight sum, as pf_narrow12 takes it
    __shared__ int32_t gg[EPI == EPI_RESID ? ITEMS : 1][EPI == EPI_RESID ? 128 : 1];
    __shared__ uint32_t silu[SILU ? 2049 : 1];
    __shared__ uint32_t last;
    // Items (row tile, part of K, output tile) of this workgroup: the items
    // of one output tile run on one XCD (workgroups go round the 8 XCDs),
    // which then reads the tile's weights from HBM once; item j0 + i stride.
    const uint32_t parts = a.parts, xcd = blockIdx.x & 7;
    const uint32_t j0 = blockIdx.x >> 3, stride = gridDim.x >> 3;
    const uint32_t njx = xcd < ntiles ? ((ntiles - xcd + 7) / 8) * parts * mtiles : 0;
    if (j0 >= njx) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave >> 1, wn = wave & 1, half = lane >> 5;
    const uint32_t S = a.steps, KC = 4 * S;
    auto item_n = [&](uint32_t j) { return j / mtiles / parts * 8 + xcd; };  // output tile
    auto item_part = [&](uint32_t j) { return j / mtiles % parts; };
    // output and matrix of slot i (0..127) of output tile ni
    auto slot_n = [&](uint32_t ni, uint32_t i) {
        return SILU ? ni * 64 + 32 * (i >> 6) + (i & 31) : ni * 128 + i;
    };
    auto slot_m = [&](uint32_t i) { return SILU ? (i >> 5) & 1 : 0u; };
    for (uint32_t i = tid >> 7; i < ITEMS && j0 + i * stride < njx; i += (NTH + 127) / 128) {
        const uint32_t sl = tid & 127, n = slot_n(item_n(j0 + i * stride), sl);
        const int32_t* ms = SILU && slot_m(sl) ? a.ms1 : a.ms0;
        const bool ok = n < a.n;
        const int32_t sum = ok ? 256 * ms[2 * n] + ms[2 * n + 1] + (WIDE ? 0 : 128 * 64 * (int32_t)a.kq) : 0;
        sw[i][sl] = WIDE ? make_int2(sum, 0) : make_int2((sum >> 1) + 8, 128 * (sum & 1) + 8);
        if (EPI == EPI_RESID)
            gg[i][sl] = ok && a.xp_out ? __mul24(a.norm_gain, (int32_t)a.norm_gamma[n]) : 0;
    }
    if (SILU)
        for (uint32_t i = tid; i < 2049; i += NTH) silu[i] = a.silu8[i];
    // weight pieces of this thread: 16 inputs of slots (q NTH + tid) / 8; a
    // wavefront's slots are of one matrix, and byte offsets fit 32 bits
    const uint32_t pc = tid & 7;
    const uint8_t* wbase[NP];
    uint32_t woff[NP], wdst[NP];
#pragma unroll
    for (int q = 0; q < NP; q++) {
        const uint32_t slot = (NTH / 8) * q + (tid >> 3);
        const bool up = SILU && __builtin_amdgcn_readfirstlane(slot_m(slot));
        wbase[q] = WIDE ? (const uint8_t*)(up ? a.mf1 : a.mf0) : (up ? a.p1 : a.p0);
        wdst[q] = (4 * (slot >> 5) + (pc >> 1)) * kWPiece + (pc & 1) * kWHalf + 16 * (slot & 31);
    }
    auto w_item = [&](uint32_t j) {  // the pieces' offsets in item j's output tile
        const uint32_t ni = item_n(j);
#pragma unroll
        for (int q = 0; q < NP; q++) {
            const uint32_t n = slot_n(ni, (NTH / 8) * q + (tid >> 3));
            if (WIDE)
                woff[q] = min(n / kMfRows, (a.n - 1) / kMfRows) * a.kq * kMfRecord +
                          (16 * (pc & 3) + n % kMfRows) * 16;
            else
                woff[q] = min(n >> 2, (a.n + 3) / 4 - 1) * S * kP12Step + 128 * (n & 3) + 16 * pc;
        }
    };
    const uint32_t noff = 512 - 64 * ((tid >> 3) & 3) - 8 * pc;  // to a piece's high nibbles
    v4u wr[2][NP];
    v4u wr2[WIDE ? 2 : 1][WIDE ? NP : 1];
    v2u wn8[WIDE ? 1 : 2][WIDE ? 1 : NP];
    auto w_load = [&](int set, uint32_t s) {
#pragma unroll
        for (int q = 0; q < NP; q++) {
            if constexpr (WIDE) {
                const uint32_t kk = 2 * s + (pc >> 2);
                const bool in = kk < a.kq;
                const uint8_t* p = wbase[q] + (woff[q] + (in ? kk : a.kq - 1) * kMfRecord);
                const uint32_t keep = lane_mask(in);
                wr[set][q] = *(const v4u*)p & v4u{keep, keep, keep, keep};
                wr2[set][q] = *(const v4u*)(p + 1024) & v4u{keep, keep, keep, keep};
            } else {
                const uint8_t* p = wbase[q] + (size_t)s * kP12Step;
                wr[set][q] = *(const v4u*)(p + woff[q]);
                wn8[set][q] = *(const v2u*)(p + (woff[q] + noff));
            }
        }
    };
    uint32_t flip = 0;  // buffer of register set 0
    auto w_store = [&](int set) {
#pragma unroll
        for (int q = 0; q < NP; q++) {
            uint8_t* d = wl + (set ^ flip) * kWBuf + wdst[q];
            if constexpr (WIDE) {
                *(v4u*)d = wr[set][q];
                *(v4u*)(d + kWPlane) = wr2[set][q];
            } else {
                v4u hi;
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const uint32_t w = e ? wn8[set][q].y : wn8[set][q].x;
                    const uint32_t x = w & 0x0F0F0F0Fu, y = (w >> 4) & 0x0F0F0F0Fu;
                    const uint32_t c0 = __builtin_amdgcn_perm(y, x, 0x06040200u);
                    const uint32_t c1 = __builtin_amdgcn_perm(y, x, 0x07050301u);
                    hi[2 * e] = p12_signed_high(c0, wr[set][q][2 * e]);
                    hi[2 * e + 1] = p12_signed_high(c1, wr[set][q][2 * e + 1]);
                }
                *(v4u*)d = hi;
                *(v4u*)(d + kWPlane) = wr[set][q];
            }
        }
    };
    v4i xb[4][2];
    // Cursors over the items' steps, the weights' and the activations' each
    // ahead of the products'; past the last step they repeat it.
    struct Cursor {
        uint32_t j, s, end;
    };
    auto first_step = [&](uint32_t j) { return item_part(j) * S / parts; };
    auto last_step = [&](uint32_t j) { return (item_part(j) + 1) * S / parts; };
    Cursor cw = {j0, first_step(j0), last_step(j0)}, cx = cw;
    const int8_t* xs = nullptr;
    auto x_item = [&](uint32_t j) { xs = a.x + (size_t)(j % mtiles * WM + wm) * KC * 2048; };
    auto advance = [&](Cursor& c) {  // whether it entered another item
        if (++c.s < c.end) return false;
        if (c.j + stride >= njx) {
            c.s--;
            return false;
        }
        c.j += stride;
        c.s = first_step(c.j);
        c.end = last_step(c.j);
        return true;
    };
    auto w_next = [&](int set) {
        w_load(set, cw.s);
        if (advance(cw)) w_item(cw.j);
    };
    auto x_load = [&](int kc) {
#pragma unroll
        for (int p = 0; p < 2; p++)
            xb[kc][p] =
                *(const v4i*)(xs + (size_t)(4 * cx.s + kc) * 2048 + 1024 * p + lane * 16);
    };
    auto x_next = [&] {
        if (advance(cx)) x_item(cx.j);
    };
    v16i acc[2][3];
    w_item(j0);
    x_item(j0);
    w_next(0);
    w_next(1);
#pragma unroll
    for (int kc = 0; kc < 4; kc++) x_load(kc);
    x_next();
    w_store(0);
    w_next(0);
    lds_barrier();
    // weight operands of piece kc of buffer b
    const uint32_t rd = 2 * wn * 4 * kWPiece + (lane & 31) * 16 + half * kWHalf;
    v4i wf[2][2][2];
    auto wf_load = [&](int set, int b, int kc) {
#pragma unroll
        for (int nt = 0; nt < 2; nt++)
#pragma unroll
            for (int p = 0; p < 2; p++)
                wf[set][nt][p] = *(const v4i*)(wl + (b ^ flip) * kWBuf + rd +
                                               (4 * nt + kc) * kWPiece + p * kWPlane);
    };
    wf_load(0, 0, 0);
    // A step from register sets and buffer P.  Piece kc's operands were read before the
    // products of the piece before it; the next step's weights go into the
    // other buffer in the middle (its last readers passed the barrier of
    // the step before), so that the barrier, before the last piece, leaves
    // products to issue behind it.  A piece's activations are reloaded for
    // the next step once used, the weights three steps on requested.
    auto step = [&](auto par) {
        constexpr int P = decltype(par)::value;
#pragma unroll
        for (int kc = 0; kc < 4; kc++) {
            const int cur = kc & 1;
            if (kc < 3) wf_load(cur ^ 1, P, kc + 1);
            else wf_load(cur ^ 1, P ^ 1, 0);
            if (kc == 1) w_store(P ^ 1);
#pragma unroll
            for (int nt = 0; nt < 2; nt++) {
                v16i* c = acc[nt];
                const v4i *w = wf[cur][nt], *x = xb[kc];
                c[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[0], x[0], c[0], 0, 0, 0);
                c[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[0], x[1], c[1], 0, 0, 0);
                c[2] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[1], x[1], c[2], 0, 0, 0);
                c[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[1], x[0], c[1], 0, 0, 0);
            }
            x_load(kc);
            if (kc == 1) w_next(P ^ 1);
            if (kc == 3) x_next();
            // keeps each piece's loads where they are: gathered at the end of
            // the step they have no products left to hide behind
            __builtin_amdgcn_sched_barrier(0);
            if (kc == 2) lds_barrier();
        }
    };
    for (uint32_t j = j0, it = 0; j < njx; j += stride, it++) {
    const uint32_t ni = item_n(j), part = item_part(j);
    const uint32_t mp = j % mtiles * WM + wm;  // this wavefront's row piece
    const uint32_t len = last_step(j) - first_step(j);
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[nt][p][i] = 0;
    for (uint32_t s = 0; s + 1 < len; s += 2) {
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
    }
    if (len & 1) {
        // the sets change places
        step(std::integral_constant<int, 0>{});
        flip ^= 1;
#pragma unroll
        for (int q = 0; q < NP; q++) {
            swap_v(wr[0][q], wr[1][q]);
            if constexpr (WIDE) swap_v(wr2[0][q], wr2[1][q]);
            else swap_v(wn8[0][q], wn8[1][q]);
        }
    }
    if (parts > 1) {
        // exact sums of this part; the last of the tile's parts to arrive
        // adds the others'
        const size_t tile = (size_t)ni * mtiles + j % mtiles;
        int64_t* base = a.part + tile * parts * (size_t)(NTH * 32) + tid;
        auto sum = [&](int i) {
            const v16i* c = acc[i >> 4];
            return ((((int64_t)c[0][i & 15] << 8) + c[1][i & 15]) << 8) + c[2][i & 15];
        };
#pragma unroll
        for (int i = 0; i < 32; i++) st_coherent(base + ((size_t)part * 32 + i) * NTH, sum(i));
        if (!arrive_last(&a.count[tile], parts, &last)) continue;
        // C sums of U parts requested together.  Left to itself the compiler
        // waits for each load before the next where a thread's registers are
        // short, two and four wavefronts: 8 us a part (down of 32 rows in
        // eight parts 79 us, 33 so); with eight it requests all 32 by itself.
        constexpr int C = WM == 4 ? 32 : 8;
        constexpr uint32_t U = WM == 4 ? 1 : 4;
#pragma unroll
        for (int i0 = 0; i0 < 32; i0 += C) {
            int64_t t[C];
#pragma unroll
            for (int i = 0; i < C; i++) t[i] = sum(i0 + i);
#pragma unroll 1
            for (uint32_t q0 = 1; q0 < parts; q0 += U) {
                int64_t o[U][C];
#pragma unroll
                for (uint32_t u = 0; u < U; u++) {
                    uint32_t q = part + (U == 1 ? q0 : min(q0 + u, parts - 1));
                    q -= q >= parts ? parts : 0;
#pragma unroll
                    for (int i = 0; i < C; i++)
                        o[u][i] = ld_coherent(base + ((size_t)q * 32 + i0 + i) * NTH);
                }
                if (WM < 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (uint32_t u = 0; u < U; u++)
#pragma unroll
                    for (int i = 0; i < C; i++) t[i] += U == 1 || q0 + u < parts ? o[u][i] : 0;
            }
#pragma unroll
            for (int i = 0; i < C; i++) {
                // back as 256 x + bd, x far outside the narrowing's range
                // where it does not fit
                constexpr int64_t lim = WIDE ? INT32_MAX : 1 << 29;
                const int64_t h = t[i] >> 8;
                v16i* c = acc[(i0 + i) >> 4];
                c[0][(i0 + i) & 15] = 0;
                c[1][(i0 + i) & 15] = (int32_t)(h < -lim ? -lim : (h > lim ? lim : h));
                c[2][(i0 + i) & 15] = (int32_t)(t[i] & 255);
            }
        }
    }
    // ---- epilogue: lane's element 4 g + t of piece nt is output 8 g + 4
    // half + t of that piece, row lane % 32 ----
    {
        int32_t rx = 0;
        if (WIDE) rx = a.rowsum[32 * mp + (lane & 31)];
        // sums of output slot `slot` (element i of piece nt) narrowed to Q8.8
        auto value = [&](int nt, int i, uint32_t slot, const uint32_t* corr) {
            const int32_t ac = acc[nt][0][i], x = acc[nt][1][i], bd = acc[nt][2][i];
            if (WIDE)
                return pf_narrow64(65536 * (int64_t)ac + 256 * (int64_t)x + bd +
                                   128 * ((int64_t)sw[it][slot].x + rx));
            int32_t sh = sw[it][slot].x, sl = sw[it][slot].y;
            if (CORR && corr && slot_n(ni, slot) < a.n) {
                // corrections of weights past 12 bits: x from its planes
                const uint4 cw = *(const uint4*)(corr + (size_t)kCorrSlots * slot_n(ni, slot));
                const uint32_t e[4] = {cw.x, cw.y, cw.z, cw.w};
                int64_t more = 0;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if ((e[q] & 0xffffu) == 0) continue;
                    const uint32_t k = e[q] >> 16;
                    const int8_t* px = a.x + ((size_t)mp * KC + k / 32) * 2048 +
                                       ((lane & 31) + 32 * ((k >> 4) & 1)) * 16 + (k & 15);
                    const int32_t xv = ((int32_t)px[0] << 8) + px[1024] + 128;
                    more += (int64_t)xv * (int16_t)(e[q] & 0xffffu);
                }
                sh += (int32_t)(more >> 8);
                sl += (int32_t)(more & 255);
            }
            return pf_narrow12(ac, x, bd, sh, sl);
        };
        // a lane's 16 int16 outputs of a piece as xp planes: halves exchange
        // so that each lane stores 16 bytes of one row
        auto store_xp = [&](const int32_t (&y)[16], uint32_t kc, uint32_t kcs) {
            uint32_t dc[4], dd[4];
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const uint32_t w0 = pack16(y[4 * g], y[4 * g + 1]);
                const uint32_t w1 = pack16(y[4 * g + 2], y[4 * g + 3]);
                dc[g] = plane_c(w0, w1);
                dd[g] = plane_d(w0, w1);
            }
            int8_t* p = a.xp_out + ((size_t)mp * kcs + kc) * 2048 + lane * 16;
#pragma unroll
            for (int pl = 0; pl < 2; pl++) {
                const uint32_t* d = pl ? dd : dc;
                const auto u = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
                const auto v = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
                *(v4u*)(p + 1024 * pl) = v4u{u[0], u[1], v[0], v[1]};
            }
        };
        if constexpr (SILU) {
            // in three passes, each over all 16 outputs: the sums narrowed
            // (which frees their registers), the table words, the products
            int32_t gate[16], up[16], y[16];
            uint32_t tw[16];
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const uint32_t sg = 64 * wn + 8 * (i >> 2) + 4 * half + (i & 3);
                gate[i] = value(0, i, sg, a.corr0);
                up[i] = value(1, i, sg + 32, a.corr1);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 16; i++) tw[i] = silu[fx_silu_index(gate[i])];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const uint32_t sg = 64 * wn + 8 * (i >> 2) + 4 * half + (i & 3);
                const int32_t sv = silu_packed(gate[i], tw[i]);
                y[i] = med3((__mul24(sv, up[i]) + 128) >> 8, INT16_MIN, INT16_MAX);
                if (slot_n(ni, sg) >= a.n) y[i] = 0;
            }
            store_xp(y, ni * 2 + wn, 2 * ntiles);
        } else {
#pragma unroll
            for (int nt = 0; nt < 2; nt++) {
                const uint32_t sl = 64 * wn + 32 * nt;
                int32_t y[16];
#pragma unroll
                for (int i = 0; i < 16; i++)
                    y[i] = value(nt, i, sl + 8 * (i >> 2) + 4 * half + (i & 3), a.corr0);
                const size_t fo = (((size_t)mp * 4 * ntiles + ni * 4 + 2 * wn + nt) * 64 + lane) * 16;
                if (EPI == EPI_RESID) {
                    const v4u r0 = *(const v4u*)(a.res + fo), r1 = *(const v4u*)(a.res + fo + 8);
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const uint32_t w = i < 8 ? r0[i >> 1] : r1[(i - 8) >> 1];
                        y[i] = sat16_32(y[i] + (int16_t)((i & 1) ? w >> 16 : w & 0xffffu));
                    }
                }
                v4u o0, o1;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    o0[i] = pack16(y[2 * i], y[2 * i + 1]);
                    o1[i] = pack16(y[8 + 2 * i], y[9 + 2 * i]);
                }
                *(v4u*)(a.out + fo) = o0;
                *(v4u*)(a.out + fo + 8) = o1;
                if (EPI == EPI_RESID && a.xp_out) {
#pragma unroll
                    for (int i = 0; i < 16; i++)
                        y[i] = norm1(y[i], gg[it][sl + 8 * (i >> 2) + 4 * half + (i & 3)]);
                    store_xp(y, ni * 4 + 2 * wn + nt, 4 * ntiles);
                }
            }
        }
    }
    }
}

__global__ __launch_bounds__(256) void pf_rowsum_kernel(const int8_t* x, uint32_t kcs,
                                                        int32_t* rowsum) {
    // thread (k part t / 32, row t % 32) of row piece blockIdx.x
    const uint32_t r = threadIdx.x & 31, part = threadIdx.x >> 5;
    int32_t s = 0;
    for (uint32_t k = part; k < 2 * kcs; k += 8) {  // half pieces
        const int8_t* p = x + ((size_t)blockIdx.x * kcs + k / 2) * 2048 + (r + 32 * (k & 1)) * 16;
        const v4i c = *(const v4i*)p, d = *(const v4i*)(p + 1024);
        int32_t sc = 0, sd = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            sc = __builtin_amdgcn_sdot4(c[i], 0x01010101, sc, false);
            sd = __builtin_amdgcn_sdot4(d[i], 0x01010101, sd, false);
        }
        s += 256 * sc + sd + 16 * 128;
    }
    __shared__ int32_t red[8][32];
    red[part][r] = s;
    __syncthreads();
    if (threadIdx.x < 32) {
        int32_t t = 0;
#pragma unroll
        for (int q = 0; q < 8; q++) t += red[q][r];
        rowsum[blockIdx.x * 32 + r] = t;
    }
}

// Thread: 16 columns of a row.
__global__ __launch_bounds__(256) void pf_init_kernel(const int16_t* rows, uint32_t m,
                                                      uint32_t cols, uint32_t kcs,
                                                      const int16_t* gamma, int32_t gain,
                                                      int16_t* h, int8_t* xp) {
    const uint32_t p = blockIdx.x * 8 + (threadIdx.x >> 5);  // 16-column group
    const uint32_t row = blockIdx.y * 32 + (threadIdx.x & 31);
    if (p >= 2 * kcs || row >= m) return;
    int32_t x[16], y[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const uint32_t n = 16 * p + i;
        const bool in = n < cols;
        x[i] = in ? rows[(size_t)row * cols + n] : 0;
        y[i] = in ? norm1(x[i], __mul24(gain, (int32_t)gamma[n])) : 0;
    }
    v4u c, d;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const uint32_t w0 = pack16(y[4 * g], y[4 * g + 1]), w1 = pack16(y[4 * g + 2], y[4 * g + 3]);
        c[g] = plane_c(w0, w1);
        d[g] = plane_d(w0, w1);
        v2u o = {pack16(x[4 * g], x[4 * g + 1]), pack16(x[4 * g + 2], x[4 * g + 3])};
        *(v2u*)(h + pf_frag16(row, 16 * p + 4 * g, kcs)) = o;
    }
    int8_t* dst = xp + ((size_t)blockIdx.y * kcs + p / 2) * 2048 +
                  ((threadIdx.x & 31) + 32 * (p & 1)) * 16;
    *(v4u*)dst = c;
    *(v4u*)(dst + 1024) = d;
}

__global__ __launch_bounds__(256) void pf_finish_kernel(
    const int16_t* h1, const int16_t* h2, uint32_t m, uint32_t cols, uint32_t k_pad,
    uint32_t block, uint32_t final_norm, const int16_t* gamma, int32_t gain, int16_t* pair0,
    int16_t* pair1) {
    const uint32_t r = blockIdx.y, n = blockIdx.x * 256 + threadIdx.x;
    if (n >= cols) return;
    const uint32_t start = (m - 1) / block * block, last = m - start;
    uint32_t t;
    if (r < last) t = start + r;
    else if (start >= block) t = start - block + r;
    else return;  // no block held such a row
    const size_t o = pf_frag16(t, n, k_pad / 32);
    const int16_t v = h2[o];
    pair1[(size_t)r * k_pad + n] = v;
    pair0[(size_t)r * k_pad + n] = final_norm && r < last
                                       ? (int16_t)norm1(v, __mul24(gain, (int32_t)gamma[n]))
                                       : h1[o];
}

// ---------------------------------------------------------------------
// Attention.  K values enter clamped to [-2048, 2048] (attn_common.h) as
// k' = 256 a + b, b a signed byte; queries as xp planes q = 256 c + d + 128;
// probabilities p = 256 c + d with d a signed byte (c <= 64); V as K.
//   q . k' = 65536 sum ac + 256 (sum ad + sum bc) + sum bd + 128 sum k'
// in units of 256, T = 256 ac + x + (L >> 8), fits int32.
// Operand pieces (16x16x64 MFMA): lane l, byte b is row (position, head
// element or query) l % 16, contraction index 16 (l / 16) + b.
// ---------------------------------------------------------------------
__device__ __forceinline__ void split_signed(int32_t v, int32_t& hi, int32_t& lo) {
    hi = (v + 128) >> 8;
    lo = v;
}
__device__ __forceinline__ uint32_t pack8(int32_t a, int32_t b, int32_t c, int32_t d) {
    return (uint32_t)(a & 255) | (uint32_t)(b & 255) << 8 | (uint32_t)(c & 255) << 16 |
           (uint32_t)(d & 255) << 24;
}

// Roles by workgroup: (KV head, tile) K pages, the same V pages, then
// (row piece of 32, query head) queries.
__global__ __launch_bounds__(256) void pf_kvq_kernel(PfAttnArgs a, uint32_t ntiles) {
    const uint32_t tid = threadIdx.x, d = a.head_dim, hd = d / 2;
    const uint32_t nkv = a.num_kv_heads * ntiles;
    const uint32_t kc64 = (d + 63) / 64;
    __shared__ __attribute__((aligned(16))) int16_t sm[64 * 136];
    if (blockIdx.x < 2 * nkv) {
        const bool isv = blockIdx.x >= nkv;
        const uint32_t id = isv ? blockIdx.x - nkv : blockIdx.x;
        const uint32_t kvh = id / ntiles, tile = id % ntiles;
        const uint32_t pg = kvh * a.tiles + tile, end = a.pos0 + a.m;
        const size_t page = (size_t)pg * TILE * d;
        const uint32_t ld = d + 8;  // LDS row of a position
        if (!isv) {
            // four pairs (e, e + d / 2) of a position at a time
            for (uint32_t i = tid; i < TILE * (hd / 4); i += 256) {
                const uint32_t p = i % TILE, e = 4 * (i / TILE), pos = tile * TILE + p;
                int32_t y0[4] = {0, 0, 0, 0}, y1[4] = {0, 0, 0, 0};
                if (pos >= end) {
                } else if (pos >= a.pos0) {
                    const uint32_t m = pos - a.pos0, n = a.num_heads * d + kvh * d + e;
                    const int16_t* rp = a.rope + (size_t)pos * d;
                    const v2u x0 = *(const v2u*)(a.qkv + pf_frag16(m, n, a.qkv_nt));
                    const v2u x1 = *(const v2u*)(a.qkv + pf_frag16(m, n + hd, a.qkv_nt));
                    const v2u cs = *(const v2u*)(rp + e), sn = *(const v2u*)(rp + hd + e);
#pragma unroll
                    for (int b = 0; b < 4; b++)
                        rope_pair(half16(x0, b), half16(x1, b), half16(cs, b), half16(sn, b), y0[b],
                                  y1[b]);
                } else {
#pragma unroll
                    for (int b = 0; b < 4; b++) {
                        y0[b] = a.kcache[page + p * d + paired(e + b)];
                        y1[b] = a.kcache[page + p * d + paired(hd + e + b)];
                    }
                }
                *(v2u*)&sm[p * ld + e] = v2u{pack16(y0[0], y0[1]), pack16(y0[2], y0[3])};
                *(v2u*)&sm[p * ld + hd + e] = v2u{pack16(y1[0], y1[1]), pack16(y1[2], y1[3])};
            }
            __syncthreads();
            for (uint32_t i = tid; i < TILE * d; i += 256) {
                const uint32_t p = i / d, s = i % d, pos = tile * TILE + p;
                if (pos >= a.pos0 && pos < end)
                    a.kcache[page + i] = sm[p * ld + (s & ~7u) + slot_pos(s & 7u)];
            }
            bool sat = false;
            int8_t* dst = a.kp + (size_t)pg * 4 * kc64 * 2048;
            for (uint32_t i = tid; i < TILE * 4 * kc64; i += 256) {
                const uint32_t p = i % TILE, g = i / TILE;  // 16-element group of row p
                int32_t hi[16], lo[16];
#pragma unroll
                for (int b = 0; b < 16; b++) {
                    const uint32_t e = 16 * g + b;
                    const int32_t k = e < d ? clamp_k(sm[p * ld + e]) : 0;
                    sat |= k == 2048;
                    split_signed(k, hi[b], lo[b]);
                }
                v4u vh, vl;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    vh[q] = pack8(hi[4 * q], hi[4 * q + 1], hi[4 * q + 2], hi[4 * q + 3]);
                    vl[q] = pack8(lo[4 * q], lo[4 * q + 1], lo[4 * q + 2], lo[4 * q + 3]);
                }
                int8_t* o = dst + ((p / 16) * kc64 + g / 4) * 2048 + (p % 16 + 16 * (g % 4)) * 16;
                *(v4u*)o = vh;
                *(v4u*)(o + 1024) = vl;
            }
            if (tid < TILE) {
                int32_t s = 0;
                for (uint32_t e = 0; e < d; e++) s += clamp_k(sm[tid * ld + e]);
                a.kbias[(size_t)pg * TILE + tid] = 128 * s;
            }
            const bool any = __syncthreads_or(sat ? 1 : 0) != 0;
            if (tid == 0) a.kvflag[pg] = any ? 1u : 0u;
        } else {
            for (uint32_t i = tid; i < TILE * (d / 4); i += 256) {
                const uint32_t p = i % TILE, e = 4 * (i / TILE), pos = tile * TILE + p;
                v2u v = {0, 0};
                if (pos >= end) {
                } else if (pos >= a.pos0) {
                    v = *(const v2u*)(a.qkv + pf_frag16(pos - a.pos0,
                                                        (a.num_heads + a.num_kv_heads) * d +
                                                            kvh * d + e, a.qkv_nt));
                } else {
                    const int16_t* q = a.vcache + page + e * TILE + paired(p);
                    v = v2u{pack16(q[0], q[TILE]), pack16(q[2 * TILE], q[3 * TILE])};
                }
                *(v2u*)&sm[p * ld + e] = v;
            }
            __syncthreads();
            for (uint32_t i = tid; i < TILE * d; i += 256) {
                const uint32_t e = i / TILE, p = (i % TILE & ~7u) + slot_pos(i & 7u);
                const uint32_t pos = tile * TILE + p;
                if (pos >= a.pos0 && pos < end) a.vcache[page + i] = sm[p * ld + e];
            }
            bool sat = false;
            const uint32_t ne = d / 16;
            int8_t* dst = a.vp + (size_t)pg * ne * 2048;
            for (uint32_t i = tid; i < 4 * d; i += 256) {
                const uint32_t e = i % d, g = i / d;  // positions 16 g .. + 15
                int32_t hi[16], lo[16];
#pragma unroll
                for (int b = 0; b < 16; b++) {
                    const int32_t v = clamp_k(sm[(16 * g + b) * ld + e]);
                    sat |= v == 2048;
                    split_signed(v, hi[b], lo[b]);
                }
                v4u vh, vl;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    vh[q] = pack8(hi[4 * q], hi[4 * q + 1], hi[4 * q + 2], hi[4 * q + 3]);
                    vl[q] = pack8(lo[4 * q], lo[4 * q + 1], lo[4 * q + 2], lo[4 * q + 3]);
                }
                int8_t* o = dst + (e / 16) * 2048 + (e % 16 + 16 * g) * 16;
                *(v4u*)o = vh;
                *(v4u*)(o + 1024) = vl;
            }
            const bool any = __syncthreads_or(sat ? 1 : 0) != 0;
            if (tid == 0) a.kvflag[a.num_kv_heads * a.tiles + pg] = any ? 1u : 0u;
        }
        return;
    }
    // ---- queries ----
    const uint32_t id = blockIdx.x - 2 * nkv, head = id % a.num_heads, mp = id / a.num_heads;
    const uint32_t mps = (a.m + 31) / 32;
    const uint32_t r = tid & 31, g = tid >> 5;  // row, 16-element group
    const uint32_t m = 32 * mp + r;
    bool extreme = false;
    if (g < 4 * kc64) {
        int32_t y[16];
        const uint32_t mr = m < a.m ? m : a.m - 1;
        const int16_t* rp = a.rope + (size_t)(a.pos0 + mr) * d;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t e = 16 * g + 4 * q;
            const bool in = e < d, lo = e < hd;  // d / 2 is a multiple of 8
            const uint32_t c = !in ? 0 : (lo ? e : e - hd), n = head * d + c;
            const v2u x0 = *(const v2u*)(a.qkv + pf_frag16(mr, n, a.qkv_nt));
            const v2u x1 = *(const v2u*)(a.qkv + pf_frag16(mr, n + hd, a.qkv_nt));
            const v2u cs = *(const v2u*)(rp + c), sn = *(const v2u*)(rp + hd + c);
#pragma unroll
            for (int b = 0; b < 4; b++) {
                int32_t y0, y1;
                rope_pair(half16(x0, b), half16(x1, b), half16(cs, b), half16(sn, b), y0, y1);
                y[4 * q + b] = !in ? 0 : (lo ? y0 : y1);
            }
        }
#pragma unroll
        for (int b = 0; b < 4; b++)
            extreme |= y[b] == -32768 && y[b + 4] == -32768 && y[b + 8] == -32768 &&
                       y[b + 12] == -32768;
        v4u c, dd;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t w0 = pack16(y[4 * q], y[4 * q + 1]);
            const uint32_t w1 = pack16(y[4 * q + 2], y[4 * q + 3]);
            c[q] = plane_c(w0, w1);
            dd[q] = plane_d(w0, w1);
        }
        int8_t* o = a.qp + (((size_t)head * mps * 2 + m / 16) * kc64 + g / 4) * 4096 +
                    (m % 16 + 16 * (g % 4)) * 16;
        *(v4u*)o = c;
        *(v4u*)(o + 1024) = dd;
        // c(q) = floor((8 - q) / 16), for keys that saturate
#pragma unroll
        for (int q = 0; q < 4; q++) {
            int32_t h[4], l[4];
#pragma unroll
            for (int t = 0; t < 4; t++) split_signed(sat_corr(y[4 * q + t]), h[t], l[t]);
            c[q] = pack8(h[0], h[1], h[2], h[3]);
            dd[q] = pack8(l[0], l[1], l[2], l[3]);
        }
        *(v4u*)(o + 2048) = c;
        *(v4u*)(o + 3072) = dd;
    }
    const bool any = __syncthreads_or(extreme ? 1 : 0) != 0;
    if (tid == 0) a.qflag[head * mps + mp] = any ? 1u : 0u;
}

__device__ __forceinline__ v4i mfma16(v4i a, v4i b, v4i c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}
// 1 in each byte whose (a, b) bytes are those of 2048 = 256 * 8 + 0.
__device__ __forceinline__ v4i mask2048(v4i a, v4i b) {
    v4i r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t z = ((uint32_t)a[i] ^ 0x08080808u) | (uint32_t)b[i];
        const uint32_t nz = ((z & 0x7f7f7f7fu) + 0x7f7f7f7fu) | z;
        r[i] = (int32_t)((~nz >> 7) & 0x01010101u);
    }
    return r;
}
// Maximum / sum over the four lanes l, l ^ 16, l ^ 32, l ^ 48.
__device__ __forceinline__ int32_t quad_max(int32_t v) {
    const auto p = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
    v = max((int32_t)p[0], (int32_t)p[1]);
    const auto q = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
    return max((int32_t)q[0], (int32_t)q[1]);
}
__device__ __forceinline__ int32_t quad_sum(int32_t v) {
    const auto p = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
    v = (int32_t)p[0] + (int32_t)p[1];
    const auto q = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
    return (int32_t)q[0] + (int32_t)q[1];
}

// One workgroup per (32 rows, query head), tiles in sequence as the
// reference's recurrence: wavefront w forms the scores of positions 16 w ..
// + 15 of the tile and the PV values of 16-element strips w, w + 4.  KC:
// 64-element chunks of a head, ES: strips per wavefront.
struct __attribute__((aligned(16))) PfAttnSmem {
    int16_t e14[2056];
    int8_t ps[2][4][1024];  // p, c(p)
    int32_t smax[32][4], ssum[32][4];
};
template <int KC, int ES, bool SLOW>
__device__ __forceinline__ void pf_attention_body(const PfAttnArgs& a, PfAttnSmem& sm) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint32_t q = lane & 15, g = lane >> 4, d = a.head_dim, ne = d / 16;
    const uint32_t mps = (a.m + 31) / 32;
    // the longest rows first
    const uint32_t head = blockIdx.x % a.num_heads, mp = mps - 1 - blockIdx.x / a.num_heads;
    const uint32_t kvh = head / a.group;
    auto& e14 = sm.e14;
    auto& ps = sm.ps;
    auto& smax = sm.smax;
    auto& ssum = sm.ssum;
    for (uint32_t i = tid; i < 257; i += 256) *(v4u*)(e14 + 8 * i) = *(const v4u*)(a.exp14 + 8 * i);
    const int32_t scale = a.qk_scale << 8;
    v4i qc[2][KC], qd[2][KC], qh[2][KC], ql[2][KC];  // q, c(q)
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
        for (int kc = 0; kc < KC; kc++) {
            const int8_t* p = a.qp + (((size_t)head * mps + mp) * 2 + rt) * KC * 4096 + kc * 4096 +
                              lane * 16;
            qc[rt][kc] = *(const v4i*)p;
            qd[rt][kc] = *(const v4i*)(p + 1024);
            qh[rt][kc] = *(const v4i*)(p + 2048);
            ql[rt][kc] = *(const v4i*)(p + 3072);
        }
    const uint32_t last = min(32 * mp + 31, a.m - 1);
    const uint32_t ntiles = (a.pos0 + last) / TILE + 1;
    int32_t own[2], mrun[2], sum[2];
    int32_t acc[ES][2][4];
#pragma unroll
    for (int rt = 0; rt < 2; rt++) {
        own[rt] = (int32_t)(a.pos0 + 32 * mp + 16 * rt + q);
        mrun[rt] = INT16_MIN;
        sum[rt] = 0;
#pragma unroll
        for (int es = 0; es < ES; es++)
#pragma unroll
            for (int s = 0; s < 4; s++) acc[es][rt][s] = 0;
    }
    const int8_t* kbase = a.kp + (size_t)kvh * a.tiles * 4 * KC * 2048 + w * KC * 2048 + lane * 16;
    const int8_t* vbase = a.vp + (size_t)kvh * a.tiles * ne * 2048 + lane * 16;
    const int32_t* bbase = a.kbias + (size_t)kvh * a.tiles * TILE + 16 * w + 4 * g;
    const uint32_t* kfl = a.kvflag + kvh * a.tiles;
    const uint32_t* vfl = kfl + a.num_kv_heads * a.tiles;
    v4i ka[KC], kb[KC], bias;
    uint32_t kf = kfl[0], vf = vfl[0];
    auto k_load = [&](uint32_t t) {
#pragma unroll
        for (int kc = 0; kc < KC; kc++) {
            const int8_t* p = kbase + (size_t)t * 4 * KC * 2048 + kc * 2048;
            ka[kc] = *(const v4i*)p;
            kb[kc] = *(const v4i*)(p + 1024);
        }
        bias = *(const v4i*)(bbase + (size_t)t * TILE);
    };
    k_load(0);
    __syncthreads();
    for (uint32_t t = 0; t < ntiles; t++) {
        v4i va[ES], vb[ES];
#pragma unroll
        for (int es = 0; es < ES; es++) {
            const uint32_t st = min(w + 4 * es, ne - 1);
            const int8_t* p = vbase + ((size_t)t * ne + st) * 2048;
            va[es] = *(const v4i*)p;
            vb[es] = *(const v4i*)(p + 1024);
        }
        // ---- scores of positions 64 t + 16 w + 4 g + s ----
        int32_t sc[2][4];
        const v4i zero = {0, 0, 0, 0};
#pragma unroll
        for (int rt = 0; rt < 2; rt++) {
            v4i mh = zero, ml = zero;  // corrections of saturating keys
            if (kf) {
#pragma unroll
                for (int kc = 0; kc < KC; kc++) {
                    const v4i mk = mask2048(ka[kc], kb[kc]);
                    mh = mfma16(mk, qh[rt][kc], mh);
                    ml = mfma16(mk, ql[rt][kc], ml);
                }
            }
            if constexpr (!SLOW) {
                v4i ac = zero, x = zero, bd = zero;
#pragma unroll
                for (int kc = 0; kc < KC; kc++) {
                    ac = mfma16(ka[kc], qc[rt][kc], ac);
                    x = mfma16(ka[kc], qd[rt][kc], x);
                    bd = mfma16(kb[kc], qd[rt][kc], bd);
                    x = mfma16(kb[kc], qc[rt][kc], x);
                }
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    // sum = 256 t + lo; the two roundings of sum * scale are
                    // floor((sum qk + 2^7 + 2^15) / 2^16) in one, and a t
                    // past 2^23 (sum past 32 bits) saturates the score
                    const int32_t l = bd[s] + bias[s] + ml[s];
                    const int32_t t = (ac[s] << 8) + x[s] + mh[s] + (l >> 8);
                    const int32_t lo = __mul24(l & 255, a.qk_scale) + 32896;
                    const int32_t v = __mul24(med3(t, -(1 << 23), (1 << 23) - 1), a.qk_scale) +
                                      (lo >> 8);
                    sc[rt][s] = med3(v >> 8, INT16_MIN, INT16_MAX);
                }
            } else {
                // a bank of 32 products may reach 2^31: the four banks
                // (elements k % 4) apart, as the reference saturates them
                int64_t tot[4] = {0, 0, 0, 0};
#pragma unroll 1
                for (uint32_t bk = 0; bk < 4; bk++) {
                    const int32_t keep = (int32_t)(0xffu << (8 * bk)), ones = 1 << (8 * bk);
                    const v4i kp4 = {keep, keep, keep, keep}, on4 = {ones, ones, ones, ones};
                    v4i ac = zero, x = zero, bd = zero, sa = zero, sb = zero, ch1 = zero, cl1 = zero;
#pragma unroll
                    for (int kc = 0; kc < KC; kc++) {
                        // an empty asm: hoisted out of the tile loop these
                        // rarely needed operands would hold registers
                        v4i c = qc[rt][kc], dd = qd[rt][kc];
                        asm volatile("" : "+v"(c), "+v"(dd));
                        c &= kp4;
                        dd &= kp4;
                        ac = mfma16(ka[kc], c, ac);
                        x = mfma16(ka[kc], dd, x);
                        bd = mfma16(kb[kc], dd, bd);
                        x = mfma16(kb[kc], c, x);
                        sa = mfma16(ka[kc], on4, sa);
                        sb = mfma16(kb[kc], on4, sb);
                        if (kf) {
                            const v4i mk = mask2048(ka[kc], kb[kc]) & kp4;
                            ch1 = mfma16(mk, qh[rt][kc], ch1);
                            cl1 = mfma16(mk, ql[rt][kc], cl1);
                        }
                    }
#pragma unroll
                    for (int s = 0; s < 4; s++) {
                        // exact modulo 2^32; only + 2^31 does not fit
                        const uint32_t v = ((uint32_t)ac[s] << 16) + ((uint32_t)x[s] << 8) +
                                           (uint32_t)bd[s] +
                                           128u * (256u * (uint32_t)sa[s] + (uint32_t)sb[s]) +
                                           256u * (uint32_t)ch1[s] + (uint32_t)cl1[s];
                        tot[s] += (int32_t)v == INT32_MIN ? (int64_t)INT32_MAX : (int64_t)(int32_t)v;
                    }
                }
#pragma unroll
                for (int s = 0; s < 4; s++)
                    sc[rt][s] = sat16_32(rnd32(rnd16_mul(fx_sat32(tot[s]), scale), 8));
            }
        }
        const uint32_t kf_n = kfl[t + 1 < ntiles ? t + 1 : t], vf_n = vfl[t + 1 < ntiles ? t + 1 : t];
        k_load(t + 1 < ntiles ? t + 1 : t);
        const int32_t p0 = (int32_t)(t * TILE + 16 * w + 4 * g);
#pragma unroll
        for (int rt = 0; rt < 2; rt++) {
            int32_t mx = INT16_MIN;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                if (p0 + s > own[rt]) sc[rt][s] = INT16_MIN;  // later positions
                mx = max(mx, sc[rt][s]);
            }
            mx = quad_max(mx);
            if (g == 0) smax[16 * rt + q][w] = mx;
        }
        lds_barrier();
        int32_t old[2];
#pragma unroll
        for (int rt = 0; rt < 2; rt++) {
            const v4i mv = *(const v4i*)smax[16 * rt + q];
            const int32_t mn = max(max(max(mv[0], mv[1]), max(mv[2], mv[3])), mrun[rt]);
            old[rt] = (int32_t)e14[max(mrun[rt] - mn, -2048) + 2048] << 2;
            mrun[rt] = mn;
            int32_t p[4], ls = 0;
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int32_t e = e14[max(sc[rt][s] - mn, -2048) + 2048];
                p[s] = p0 + s <= own[rt] ? e : 0;
                ls += p[s];
            }
            const uint32_t w0 = pack16(p[0], p[1]), w1 = pack16(p[2], p[3]);
            const uint32_t lane_off = (q + 16 * w) * 16 + 4 * g;
            // p + 128 <= 16512: no carry between the halves
            *(uint32_t*)&ps[rt][0][lane_off] = plane_c(w0 + 0x00800080u, w1 + 0x00800080u);
            *(uint32_t*)&ps[rt][1][lane_off] = __builtin_amdgcn_perm(w1, w0, 0x06040200u);
            if (vf) {
                // c(p) in [-1024, 0] (p = 16384 has (8 - 16384) >> 4), as 256 h + l
                const uint32_t u0 = pack16(sat_corr(p[0]), sat_corr(p[1]));
                const uint32_t u1 = pack16(sat_corr(p[2]), sat_corr(p[3]));
                *(uint32_t*)&ps[rt][3][lane_off] = __builtin_amdgcn_perm(u1, u0, 0x06040200u);
                *(uint32_t*)&ps[rt][2][lane_off] = plane_c(
                    pack16(sat_corr(p[0]) + 128, sat_corr(p[1]) + 128),
                    pack16(sat_corr(p[2]) + 128, sat_corr(p[3]) + 128));
            }
            ls = quad_sum(ls);
            if (g == 0) ssum[16 * rt + q][w] = ls;
        }
        lds_barrier();
        v4i pc[2], pd[2], ph[2], pl[2];
#pragma unroll
        for (int rt = 0; rt < 2; rt++) {
            ph[rt] = pl[rt] = zero;
            if (vf) {
                ph[rt] = *(const v4i*)&ps[rt][2][lane * 16];
                pl[rt] = *(const v4i*)&ps[rt][3][lane * 16];
            }
            pc[rt] = *(const v4i*)&ps[rt][0][lane * 16];
            pd[rt] = *(const v4i*)&ps[rt][1][lane * 16];
            const v4i sv = *(const v4i*)ssum[16 * rt + q];
            const int32_t tsum = (sv[0] + sv[1] + sv[2] + sv[3]) << 2;
            sum[rt] = __builtin_elementwise_add_sat(rnd16_mul(sum[rt], old[rt]), tsum);
        }
        // ---- PV of strips w, w + 4: element 16 strip + 4 g + s ----
        if (__any(old[0] != 65536 || old[1] != 65536)) {  // else the factors are 1.0
#pragma unroll
            for (int es = 0; es < ES; es++)
#pragma unroll
                for (int rt = 0; rt < 2; rt++)
#pragma unroll
                    for (int s = 0; s < 4; s++)
                        acc[es][rt][s] = rnd16_mul(acc[es][rt][s], old[rt]);
        }
#pragma unroll
        for (int es = 0; es < ES; es++) {
#pragma unroll
            for (int rt = 0; rt < 2; rt++) {
                v4i ac = mfma16(va[es], pc[rt], zero);
                v4i x = mfma16(va[es], pd[rt], zero);
                v4i bd = mfma16(vb[es], pd[rt], zero);
                x = mfma16(vb[es], pc[rt], x);
                if (vf) {
                    const v4i mk = mask2048(va[es], vb[es]);
                    x = mfma16(mk, ph[rt], x);
                    bd = mfma16(mk, pl[rt], bd);
                }
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    // sums in [-2^31, 2^31 - 2^16] (64 products of at most 2^14
                    // and -2048, or 2048 with its correction of -1024): exact
                    // in 32 bits, and so with 8224 added
                    const uint32_t tot = ((((uint32_t)ac[s] << 8) + (uint32_t)x[s]) << 8) +
                                         (uint32_t)bd[s];
                    // rnd(rnd(tot, 6), 8) = floor((tot + 2^5 + 2^13) / 2^14)
                    const int32_t tv = med3((int32_t)(tot + 8224) >> 14, INT16_MIN, INT16_MAX);
                    acc[es][rt][s] = __builtin_elementwise_add_sat(acc[es][rt][s], tv << 8);
                }
            }
        }
        kf = kf_n;
        vf = vf_n;
    }
    // ---- outputs as xp planes: input 16 (head d / 16 + strip) + 4 g + s ----
#pragma unroll
    for (int rt = 0; rt < 2; rt++) {
        const int32_t inv = fx_inv_sum(sum[rt]);
        const uint32_t m = 32 * mp + 16 * rt + q;
#pragma unroll
        for (int es = 0; es < ES; es++) {
            const uint32_t st = w + 4 * es;
            if (st >= ne || m >= a.m) continue;
            int32_t y[4];
#pragma unroll
            for (int s = 0; s < 4; s++) y[s] = sat16_32(rnd16_mul(acc[es][rt][s], inv));
            const uint32_t w0 = pack16(y[0], y[1]), w1 = pack16(y[2], y[3]);
            const uint32_t kg = head * ne + st;  // 16-input group
            int8_t* o = a.xp_out + ((size_t)mp * 4 * a.out_steps + kg / 2) * 2048 +
                        (m % 32 + 32 * (kg & 1)) * 16 + 4 * g;
            *(uint32_t*)o = plane_c(w0, w1);
            *(uint32_t*)(o + 1024) = plane_d(w0, w1);
        }
    }
}

template <int KC, int ES>
__global__ __launch_bounds__(256, 2) void pf_attention_kernel(PfAttnArgs a) {
    __shared__ PfAttnSmem sm;
    const uint32_t mps = (a.m + 31) / 32;
    const uint32_t head = blockIdx.x % a.num_heads, mp = mps - 1 - blockIdx.x / a.num_heads;
    if (a.qflag[head * mps + mp] == 0)
        pf_attention_body<KC, ES, false>(a, sm);
    else
        pf_attention_body<KC, ES, true>(a, sm);
}

template <int WM, int EPI>
hipError_t pf_gemm(const PfGemmArgs& a, uint32_t ntiles, hipStream_t st) {
    const uint32_t mtiles = (a.m + 32 * WM - 1) / (32 * WM);
    // items of the fullest XCD; a workgroup of four row pieces, one per
    // compute unit, takes several in turn (at most kPfItems)
    const uint32_t items = mtiles * a.parts * ((ntiles + 7) / 8);
    uint32_t wgs = items;
    if (WM == 4) wgs = std::max(std::min(items, 32u), (items + kPfItems - 1) / kPfItems);
    const dim3 g(8 * wgs), b(128 * WM);
    if (!a.p0)
        hipLaunchKernelGGL((pf_gemm_kernel<WM, EPI, true, false>), g, b, 0, st, a, mtiles, ntiles);
    else if (a.corr0 || a.corr1)
        hipLaunchKernelGGL((pf_gemm_kernel<WM, EPI, false, true>), g, b, 0, st, a, mtiles, ntiles);
    else
        hipLaunchKernelGGL((pf_gemm_kernel<WM, EPI, false, false>), g, b, 0, st, a, mtiles, ntiles);
    return hipGetLastError();
}

template <int EPI>
hipError_t pf_gemm_w(const PfGemmArgs& a, uint32_t ntiles, uint32_t wm, hipStream_t st) {
    switch (wm) {
    case 1: return pf_gemm<1, EPI>(a, ntiles, st);
    case 2: return pf_gemm<2, EPI>(a, ntiles, st);
    default: return pf_gemm<4, EPI>(a, ntiles, st);
    }
}

}  // namespace

// Row pieces per workgroup: the fewest that hold the rows, at most four (the
// weights of a workgroup are unpacked once for all of them).  K is split
// while the tiles alone leave half of the 256 compute units idle: the parts'
// exchange takes ~15 us on a full chip, a 128-input step ~1.5 us, so at least
// 32 steps stay with a part there (down, 1,024 rows, 86 steps: 137 us whole,
// 85 in two parts; Q|K|V, 16 steps: 33 and 47).  Where it is nearly empty, 8
// steps (128 rows, Q|K|V in 8 and in 4 steps a part: 26 us both) or, with the
// smaller exchange of at most 64 rows, 4 (32 rows, O in two and four parts:
// 25 and 21 us, Q|K|V 24 and 20; of 2 steps 22).
PfShape pf_gemm_shape(uint32_t m, uint32_t n, uint32_t steps, int epi) {
    const uint32_t ntiles = epi == EPI_SILU ? (n + 127) / 128 * 2 : (n + 127) / 128;
    PfShape s;
    s.wm = m <= 32 ? 1 : (m <= 64 ? 2 : 4);
    s.tiles = ntiles * ((m + 32 * s.wm - 1) / (32 * s.wm));
    s.parts = 1;
    while (s.parts < 8 && 2 * s.tiles * s.parts <= 256 &&
           steps / (2 * s.parts) >= (s.tiles * s.parts >= 128 ? 32u : s.wm == 4 ? 8u : 4u))
        s.parts *= 2;
    return s;
}

hipError_t launch_pf_gemm(const PfGemmArgs& a0, int epi, hipStream_t st) {
    if (a0.m == 0 || a0.steps == 0 || a0.steps > kP12MaxSteps || a0.n % 4)
        return hipErrorInvalidValue;
    PfGemmArgs a = a0;
    const PfShape sh = pf_gemm_shape(a.m, a.n, a.steps, epi);
    a.parts = sh.parts;
    if (sh.parts > 1 && (sh.tiles > a.max_tiles || pf_part_bytes(sh) > a.part_bytes)) a.parts = 1;
    const uint32_t ntiles = epi == EPI_SILU ? (a.n + 127) / 128 * 2 : (a.n + 127) / 128;
    switch (epi) {
    case EPI_STORE: return pf_gemm_w<EPI_STORE>(a, ntiles, sh.wm, st);
    case EPI_RESID: return pf_gemm_w<EPI_RESID>(a, ntiles, sh.wm, st);
    case EPI_SILU: return pf_gemm_w<EPI_SILU>(a, ntiles, sh.wm, st);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_pf_rowsum(const int8_t* x, uint32_t m, uint32_t steps, int32_t* rowsum,
                            hipStream_t st) {
    hipLaunchKernelGGL(pf_rowsum_kernel, dim3((m + 31) / 32), dim3(256), 0, st, x, 4 * steps, rowsum);
    return hipGetLastError();
}

hipError_t launch_pf_init(const int16_t* rows, uint32_t m, uint32_t cols, uint32_t k_pad,
                          const int16_t* gamma, int32_t gain, int16_t* h, int8_t* xp,
                          hipStream_t st) {
    hipLaunchKernelGGL(pf_init_kernel, dim3((k_pad / 16 + 7) / 8, (m + 31) / 32), dim3(256), 0, st,
                       rows, m, cols, k_pad / 32, gamma, gain, h, xp);
    return hipGetLastError();
}

size_t pf_qp_bytes(uint32_t rows_pad, uint32_t heads, uint32_t d) {
    return (size_t)heads * (rows_pad / 16) * ((d + 63) / 64) * 4096;
}
size_t pf_kp_bytes(uint32_t kv_heads, uint32_t tiles, uint32_t d) {
    return (size_t)kv_heads * tiles * 4 * ((d + 63) / 64) * 2048;
}
size_t pf_vp_bytes(uint32_t kv_heads, uint32_t tiles, uint32_t d) {
    return (size_t)kv_heads * tiles * (d / 16) * 2048;
}

hipError_t launch_pf_kvq(const PfAttnArgs& a, hipStream_t st) {
    const uint32_t nt = (a.pos0 + a.m + TILE - 1) / TILE;
    const uint32_t grid = 2 * a.num_kv_heads * nt + a.num_heads * ((a.m + 31) / 32);
    hipLaunchKernelGGL(pf_kvq_kernel, dim3(grid), dim3(256), 0, st, a, nt);
    return hipGetLastError();
}

hipError_t launch_pf_attention(const PfAttnArgs& a, hipStream_t st) {
    const uint32_t grid = a.num_heads * ((a.m + 31) / 32);
    if (a.head_dim % 16 || a.head_dim > 128) return hipErrorInvalidValue;
    if (a.head_dim > 64)
        hipLaunchKernelGGL((pf_attention_kernel<2, 2>), dim3(grid), dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((pf_attention_kernel<1, 1>), dim3(grid), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_pf_finish(const int16_t* h1, const int16_t* h2, uint32_t m, uint32_t cols,
                            uint32_t k_pad, uint32_t block, bool final_norm,
                            const int16_t* gamma, int32_t gain, int16_t* pair0, int16_t* pair1,
                            hipStream_t st) {
    hipLaunchKernelGGL(pf_finish_kernel, dim3((cols + 255) / 256, block), dim3(256), 0, st, h1, h2,
                       m, cols, k_pad, block, final_norm ? 1u : 0u, gamma, gain, pair0, pair1);
    return hipGetLastError();
}

}  // namespace llm
