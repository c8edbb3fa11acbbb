// The prompt matmul for Q4_K rows: Y[t] = W x_t for batches past 16 tokens
// (the reference's matmul_big path for prompts, engine/src/vk_backend.cpp:
// 866-918; its CPU restatement engine/src/cpu_backend.cpp:18-41).
//
// fp16 matrix cores with exact operands. A Q4_K weight is d*sc_s*q - dmin*m_s
// (q 0..15, sc_s and m_s 6-bit per 32-value sub-block s; quants.cpp:133-160),
// so per 256-value block
//   y += d * sum_s sum_k (sc_s q_k) x_k  -  dmin * sum_s m_s X_s
// with X_s the sub-block's sum of x. Both inner sums run on the matrix cores:
//  * sc_s q <= 945 is an exact fp16 integer, so the weight operand carries the
//    sub-block scale and one fp32 accumulator P collects all 8 sub-blocks of a
//    block (16 v_mfma_f32_16x16x32_f16 per 16x16 tile and block);
//  * the activations arrive as two fp16 planes of x 2^-e (hi + lo, about 22
//    bits; the per-token power of two keeps the residual stream's 1e11-sized
//    values in range), each multiplied into P by its own MFMA;
//  * the min term is one v_mfma_f32_16x16x16_f16 per tile and block: lane
//    group k (of 4) carries (m_2k, m_2k+1, m_2k, m_2k+1) against the hi and lo
//    halves of (X_2k, X_2k+1) / 32.
// Per block and output only y += d P - 32 dmin Q is left for the VALU, and
// y = acc 2^e at the end.
//
// Lane layout of the 16x16x32 MFMA: A lane l = token l%16, k-group l/16 (8
// values); B lane l = weight row l%16, the same k-group; D lane l = tokens
// 4*(l/16)+i of row l%16 (16x16x16: 4 values per k-group, the same D), so a
// lane needs only its own row's d and dmin. The k order inside an MFMA only
// has to agree between A and B: k-group k takes sub-blocks 2k and 2k + 1 of
// the block, whose 64 quants are 32 consecutive bytes of the row and whose
// scales are the only ones the lane decodes, once per block. Stage S (of 4)
// of a block is quant bytes 8 S .. 8 S + 7 of every k-group: low nibbles
// (sub-block 2k) one MFMA step, high nibbles (2k + 1) the next. The
// activation records (hact_*) are stored in that order.
//
// Workgroup: RG waves, each RT row tiles of 16 (GLU: half of gate, half of up)
// x TT token tiles of 16. LDS holds four stages of activations (32
// values of every token: TOK x 128 bytes), two blocks of the weight rows (144
// bytes a row, as stored) and of the tokens' sums, all brought in by DMA
// (global_load_lds_*) two stages or a block ahead; a wave's DMA source offsets are
// fixed per lane, and the loop issues no register loads, so the only waits on
// memory are the explicit vmcnt ones. A token's 8 pieces of 16 bytes per
// stage sit at piece ^ (token / 2 & 7), so the 16 lanes that read one piece of
// 16 tokens hit 16 different bank groups; 144-byte rows do so by themselves.
// Split-K (whole blocks) when rows x tokens alone give too few workgroups; a
// second kernel adds the partial sums in a fixed order.
//
// What bounds it: per 64 values a wave issues 68 MFMAs (1088 cycles of the
// matrix core, 544 of them also of the vector ALU) and about 95 vector
// instructions (380 cycles), two waves a SIMD; the loop takes about 1.6 times
// the matrix core's time, at 2.2 GHz. It was twice that with the pieces read
// right before their MFMAs. Gate/up of 256 tokens, 14336 x 4096: 152 us before
// (64 of gate and up a 4-wave workgroup, two a CU, LDS reads and the unpack in
// front of the MFMAs), 114-121 us now, run to run (497-527 TFLOP/s of useful
// products, twice that issued); down 86 -> 57-59 us, QKV 54 -> 32-36 us, wo 37 ->
// 23-24 us, the last three also by the outputs' way through LDS. 64 weight rows a wave (half the LDS
// reads) measured slower: four waves of 64 rows x 128 tokens 138 us, eight of 64
// x 64 151 us (their unpack is made twice, or no second wave hides the waits).
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace ts5hip {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));

struct WideArgs {
    const uint8_t *w, *w2;  // Q4_K rows (w2: GLU's up projection)
    const uint8_t *act;     // M records of hact_bytes(n_in)
    int64_t act_stride;
    float *out;             // ks == 1: y [M][ldy]; ks > 1: partials [ks][2][M][nrows]
    const float *y_in;      // W_ADD: residual [M][ldy] (may be out)
    int64_t ldy;
    int nrows, nb, n_in, M, ks;
    int units, ntt;         // (row tile, split) units; token tiles of each
    int gelu;               // W_GLU: GELU (tanh form) for SiLU
};

enum { W_STORE = 0, W_ADD = 1, W_GLU = 2 };

template <int MODE_, int RT_, int TT_, int RG_>
struct WideShape {
    static constexpr int MODE = MODE_, RT = RT_, TT = TT_, RG = RG_, NT = 64 * RG;
    static constexpr int WROWS = 16 * RT * RG, ROWS = MODE == W_GLU ? WROWS / 2 : WROWS;  // weight rows, output rows
    static constexpr int TOK = 16 * TT;
    static constexpr int PB = TOK * 8 / RG, NB = (PB + 63) / 64;        // activation pieces (16 bytes) a wave and stage, DMAs
    static constexpr int PW = 16 * RT * 9, NWI = (PW + 63) / 64;   // weight pieces a wave and block, DMAs
    static constexpr int PX = TOK * 2 / RG;                             // sum pieces a wave and block (one DMA)
    static_assert(TOK * 8 % RG == 0 && PX <= 64 && RT % 2 == 0, "wide matmul shape");
};
template <class SH>
struct WideLds {
    uint4 b[4][SH::TOK * 8];     // [token][piece ^ (token / 2 & 7)]: hi pieces of the 4 k-groups, then lo
    uint4 w[2][SH::WROWS * 9];   // [row group][row]: the row's 144-byte block
    uint4 x[2][SH::TOK * 2];     // [token][k-group]: (hi_0, hi_1), (lo_0, lo_1) of its sub-blocks' sums / 32
};
// Over the same space at the end: the tile's outputs, 4 floats between tokens'
// rows so that the lane groups of an MFMA result hit different banks.
template <class SH>
struct WideOut {
    float y[SH::TOK][SH::WROWS + 4];
};
template <class SH>
union WideSpace {
    WideLds<SH> in;
    WideOut<SH> out;
};

__device__ inline void dma16s(const uint8_t *sbase, uint32_t voff, uint32_t lds_base) {
    asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "{m0}"(lds_base) : "memory");
}

// A row's block header, as the lane needs it: the scales and mins of its two
// sub-blocks (bytes sc_0, sc_1, m_0, m_1) and the (d, dmin) halves.
struct WideHdr {
    uint32_t sm, dd;
};
__device__ inline WideHdr wide_hdr(uint4 h, int kq) {
    const int s = 16 * (kq & 1);
    const uint32_t A = h.y >> s, B = h.z >> s, C = h.w >> s;
    const uint32_t split = 0u - (uint32_t)(kq >> 1);  // sub-blocks 4-7: low 4 bits from C, top 2 from A or B
    const uint32_t sc = (((C & 0x0F0Fu) | ((A >> 2) & 0x3030u)) & split) | (A & 0x3F3Fu & ~split);
    const uint32_t m = ((((C >> 4) & 0x0F0Fu) | ((B >> 2) & 0x3030u)) & split) | (B & 0x3F3Fu & ~split);
    return WideHdr{sc | m << 16, h.x};
}
// Bytes `sel` (two) of v as fp16 integers: 0x64bb is 1024 + b.
__device__ inline v2h bytes_f16(uint32_t v, uint32_t sel) {
    return __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, v, sel)) - v2h{(_Float16)1024, (_Float16)1024};
}

// A wave's registers over the K loop.
template <class SH>
struct WideRegs {
    v4f acc[SH::RT][SH::TT];      // tokens 4 kq + i of the lane's row
    v4f P[SH::RT][SH::TT];        // the block's sum of sc q x
    v4f Q[SH::RT / 2];            // half the row tiles' sums of m X / 32, of one token tile
    WideHdr hd[SH::RT], hn[SH::RT];  // the row's header, this block's and the next's
    uint2 q[SH::RT];              // the lane's 8 quant bytes of a pair of stages
    v2h sc[SH::RT], off[SH::RT];  // (sc_0, sc_1), (-1024 sc_0, -64 sc_1)
    v8h W[2][SH::RT];             // the weights of a stage's low and high nibbles
    v8h f[4];                     // the activations of the next tile steps, a ring
};
// The lane's quants of stages 2 S and 2 S + 1 from LDS (`wl`: its first row's block).
template <class SH>
__device__ inline void wide_read_q(const uint8_t *wl, WideRegs<SH> &R, int S, int kq) {
#pragma unroll
    for (int p = 0; p < SH::RT; p++) R.q[p] = *(const uint2 *)(wl + p * 16 * Q4K_BYTES + 16 + 32 * kq + 8 * S);
}
template <class SH>
__device__ inline void wide_scales(WideRegs<SH> &R, int p) {
    R.hd[p] = R.hn[p];
    R.sc[p] = bytes_f16(R.hd[p].sm, 0x04010400u);
    R.off[p] = R.sc[p] * v2h{(_Float16)-1024, (_Float16)-64};
}
// Masks and magics of the nibble unpack, opaque to the compiler so that each
// stays in a register and `and` and `or` become one instruction.
struct WideConst {
    uint32_t mask[2], magic[2];
};
__device__ inline WideConst wide_const() {
    WideConst k;
    asm("v_mov_b32 %0, 0x000F000F" : "=v"(k.mask[0]));
    asm("v_mov_b32 %0, 0x00F000F0" : "=v"(k.mask[1]));
    asm("s_mov_b32 %0, 0x64006400" : "=s"(k.magic[0]));
    asm("s_mov_b32 %0, 0x54005400" : "=s"(k.magic[1]));
    return k;
}
// Pair u (row tile u / 4, pair u % 4 of its 8 values) of the weights of step c:
// the low (0) or high (1) nibbles of bytes 0 and 2, 1 and 3, 4 and 6, 5 and 7
// (the activations' order within 8 values) times the sub-block scale, as exact
// fp16 integers (q sc <= 945). 0x640q is 1024 + q, 0x54q0 is 64 + q;
// fma(1024 + q, sc, -1024 sc) rounds once, to the exact q sc.
template <class SH>
__device__ inline void wide_pair(WideRegs<SH> &R, const WideConst &K, int u, int c) {
    const int p = u / 4, k = u % 4;
    const uint32_t d = k < 2 ? R.q[p].x : R.q[p].y, v = (k & 1) ? d >> 8 : d;
    const v2h n = __builtin_bit_cast(v2h, (v & K.mask[c]) | K.magic[c]);
    const v2h w = __builtin_elementwise_fma(n, v2h{R.sc[p][c], R.sc[p][c]}, v2h{R.off[p][c], R.off[p][c]});
    R.W[c][p][2 * k] = w[0], R.W[c][p][2 * k + 1] = w[1];
}

// Stage I = 2 S + c of a block: tile step j = (token tile g, plane) is one
// piece per lane and RT MFMAs. Pieces are read from LDS 3 steps ahead of their
// MFMAs, the last ones from the next stage, and the next stage's weights are
// made beside this one's MFMAs: a 16 x 16 x 32 MFMA holds the matrix core for 16
// cycles and the vector ALU for 8, so two vector instructions beside each are
// free and every further one costs its 4 cycles; they are spread evenly, and
// nothing but the barrier stands between two stages. `bl`: the lane's first
// piece place in slot 0; `wl`, `wn`: its first row's block in LDS, this block's
// and the next's; `xl`: the block's sums of its token (first tile).
template <class SH, int I>
__device__ __forceinline__ void wide_stage(const uint8_t *wl, const uint8_t *wn, const uint8_t *const (&bl)[2],
                                           const uint8_t *xl, WideRegs<SH> &R, const WideConst &K, int kq) {
    constexpr int RT = SH::RT, TT = SH::TT, S = I / 2, c = I % 2, NJ = 2 * TT, NPAIR = 4 * RT;
    constexpr int F0 = I * NJ;  // the ring's phase (8 NJ steps a block: a multiple of 4)
    constexpr bool last = I == 7;
    auto load = [&](int j) {
        const int slot = (j < NJ ? I : I + 1) & 3, g = j % NJ / 2, pl = j & 1;
        R.f[(F0 + j) & 3] = *(const v8h *)(bl[pl] + slot * (SH::TOK * 128) + 2048 * g);
    };
    float d[RT], dmin[RT];
    v2h amin[RT];
    // Block end: acc += d P - 32 dmin Q with Q = sum(m X / 32), for half the row
    // tiles of one token tile a step: Q half 0 of tile g is made in step (g, pl
    // 1), half 1 in the step after; each half is finished a step after its Q.
    auto mins = [&](int g, int half, uint2 x) {
#pragma unroll
        for (int i = 0; i < RT / 2; i++) {
            const v2h m = amin[half * RT / 2 + i];
            R.Q[i] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(v4h, x), v4h{m[0], m[1], m[0], m[1]},
                                                           v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        }
    };
    auto finish = [&](int g, int half) {
#pragma unroll
        for (int i = 0; i < RT / 2; i++) {
            const int p = half * RT / 2 + i;
#pragma unroll
            for (int e = 0; e < 4; e++)
                R.acc[p][g][e] = fmaf(d[p], R.P[p][g][e], fmaf(-dmin[p], R.Q[i][e], R.acc[p][g][e]));
        }
    };
    uint2 xq[2];
    uint4 h[RT];
    if constexpr (last) {
#pragma unroll
        for (int p = 0; p < RT; p++)
            amin[p] = bytes_f16(R.hd[p].sm, 0x04030402u), d[p] = h2f(R.hd[p].dd & 0xffff),
            dmin[p] = 32.0f * h2f(R.hd[p].dd >> 16);
    }
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int g = j / 2, pl = j & 1;
        load(j + 3);
        if (j == 0 && I == 6)
#pragma unroll
            for (int p = 0; p < RT; p++) h[p] = *(const uint4 *)(wn + p * 16 * Q4K_BYTES);
        if (last && pl == 0) xq[g & 1] = *(const uint2 *)(xl + 512 * g);
        if (j == 0 && c == 1) wide_read_q<SH>(last ? wn : wl, R, last ? 0 : S + 1, kq);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < RT; p++) {
            const v4f c0 = (I == 0 && pl == 0) ? v4f{0.f, 0.f, 0.f, 0.f} : R.P[p][g];
            R.P[p][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(R.f[(F0 + j) & 3], R.W[c][p], c0, 0, 0, 0);
        }
        // The next stage's weights, over all tile steps, or all but the first
        // two where their quants (and the next block's scales) come first.
        constexpr int J0 = c == 1 ? 2 : 0, n = NJ - J0;
        if (last && j < J0)
#pragma unroll
            for (int p = 0; p < RT; p++)
                if (p * J0 / RT == j) wide_scales<SH>(R, p);
        if (j >= J0)
#pragma unroll
            for (int u = (j - J0) * NPAIR / n; u < (j - J0 + 1) * NPAIR / n; u++) wide_pair<SH>(R, K, u, 1 - c);
        if (I == 6 && j >= NJ - RT) R.hn[j - (NJ - RT)] = wide_hdr(h[j - (NJ - RT)], kq);  // the next block's headers
        if (last) {
            if (j > 1) finish((j - 2) / 2, pl);
            if (pl == 1) mins(g, 0, xq[g & 1]);
            else if (g > 0) mins(g - 1, 1, xq[(g - 1) & 1]);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (last) {
        finish(TT - 1, 0);
        mins(TT - 1, 1, xq[(TT - 1) & 1]);
        finish(TT - 1, 1);
    }
}

template <class SH>
__global__ __launch_bounds__(SH::NT, 2) void k_gemm_wide(WideArgs a) {
    constexpr int MODE = SH::MODE, RT = SH::RT, TT = SH::TT;
    constexpr int RTM = MODE == W_GLU ? RT / 2 : RT;  // row tiles per matrix and wave
    __shared__ WideSpace<SH> space;
    __shared__ __align__(16) float us[SH::TOK];  // the tokens' 2^e
    WideLds<SH> &L = space.in;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, kq = lane >> 4, rl = lane & 15;
    // Workgroups go to the 8 XCDs in turn: the token tiles of one unit (row
    // tile, split) follow each other on one XCD, whose L2 then serves the
    // weights to all but the first.
    const int id = blockIdx.x, jx = id >> 3;
    const int unit = (jx / a.ntt) * 8 + (id & 7);
    if (unit >= a.units) return;
    const int t0 = (jx % a.ntt) * SH::TOK, row0 = (unit / a.ks) * SH::ROWS, rw = row0 + 16 * RTM * wave, z = unit % a.ks;
    const int bps = (a.nb + a.ks - 1) / a.ks, bk0 = z * bps;
    const int nblk = max(0, min(a.nb, bk0 + bps) - bk0);

    uint32_t oact[SH::NB];
#pragma unroll
    for (int i = 0; i < SH::NB; i++) {
        const int u = SH::PB * wave + min(64 * i + lane, SH::PB - 1), tok = u >> 3, p = (u & 7) ^ ((tok >> 1) & 7);
        oact[i] = (uint32_t)((min(t0 + tok, a.M - 1) - t0) * a.act_stride) + p * 16;
    }
    const int xu = SH::PX * wave + min(lane, SH::PX - 1);
    const uint32_t ox = (uint32_t)((min(t0 + (xu >> 1), a.M - 1) - t0) * a.act_stride) + 16 * (xu & 1);
    const uint8_t *wp[SH::NWI];  // weight pieces of block 0: piece u is 16 bytes u % 9 of the wave's row u / 9 (clamped)
#pragma unroll
    for (int i = 0; i < SH::NWI; i++) {
        const int u = min(64 * i + lane, SH::PW - 1), lr = u / 9, p = lr >> 4;
        const int row = min(rw + 16 * (p % RTM) + (lr & 15), a.nrows - 1);
        wp[i] = (MODE == W_GLU && p / RTM ? a.w2 : a.w) + (int64_t)row * a.nb * Q4K_BYTES + 16 * (u % 9);
    }
    const uint8_t *act_base = a.act + (int64_t)t0 * a.act_stride;
    const uint8_t *x_base = act_base + hact_x(a.n_in);

    auto issue_b = [&](int b, int I) {  // stage I of block b -> slot I mod 4
        const uint8_t *ab = act_base + (int64_t)b * 1024 + I * 128;
        const uint32_t to = lds_addr(&L.b[I & 3][SH::PB * wave]);
#pragma unroll
        for (int i = 0; i < SH::NB; i++)
            if (64 * (i + 1) <= SH::PB || lane < SH::PB - 64 * i) dma16s(ab, oact[i], to + 1024 * i);
    };
    auto issue_w = [&](int b, int buf) {  // block b's weights and sums -> w[buf], x[buf]: NWI + 1 DMAs
        const uint32_t wb = lds_addr(&L.w[buf][wave * RT * 16 * 9]);
#pragma unroll
        for (int i = 0; i < SH::NWI; i++)
            if (64 * (i + 1) <= SH::PW || lane < SH::PW - 64 * i) dma16(wp[i] + (int64_t)b * Q4K_BYTES, wb + 1024 * i);
        if (SH::PX == 64 || lane < SH::PX) dma16s(x_base + (int64_t)b * 32, ox, lds_addr(&L.x[buf][SH::PX * wave]));
    };

    WideRegs<SH> R;
#pragma unroll
    for (int p = 0; p < RT; p++)
#pragma unroll
        for (int g = 0; g < TT; g++) R.acc[p][g] = v4f{0.f, 0.f, 0.f, 0.f};

    const uint8_t *tb = (const uint8_t *)L.b[0] + rl * 128;
    const uint8_t *const bl[2] = {tb + 16 * (kq ^ (rl >> 1)), tb + 16 * ((4 + kq) ^ (rl >> 1))};
    const uint8_t *wr[2], *xr[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        wr[i] = (const uint8_t *)&L.w[i][(wave * RT * 16 + rl) * 9];
        xr[i] = (const uint8_t *)L.x[i] + rl * 32 + 8 * kq;
    }
    const WideConst K = wide_const();
    // At a stage's start every wave waits for its own DMA of the next stage,
    // issued two stages ago; the barrier then makes all of it visible and
    // frees the slot of the stage before, into which the stage after next but
    // one goes. A block's weights and sums are issued in stage 0 of the block
    // before, behind that stage's activations, and are waited for in stage 3.
    constexpr int NB = SH::NB, NW = SH::NWI + 1;  // DMAs of a stage, of a block
    auto sync = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    if (64 * wave < SH::TOK && 64 * wave + lane < SH::TOK)
        dma4(act_base + (int64_t)(min(t0 + 64 * wave + lane, a.M - 1) - t0) * a.act_stride + hact_unscale(a.n_in),
             lds_addr(&us[64 * wave]));
    if (nblk > 0) {
        issue_w(bk0, 0);
        issue_b(bk0, 0);
        issue_b(bk0, 1);
        issue_b(bk0, 2);
        wait_vm_n<2 * NB>();
        sync();
#pragma unroll
        for (int p = 0; p < RT; p++) R.hn[p] = wide_hdr(*(const uint4 *)(wr[0] + p * 16 * Q4K_BYTES), kq);
        wide_read_q<SH>(wr[0], R, 0, kq);
#pragma unroll
        for (int j = 0; j < 3; j++) R.f[j] = *(const v8h *)(bl[j & 1] + 2048 * (j / 2));
#pragma unroll
        for (int p = 0; p < RT; p++) wide_scales<SH>(R, p);
#pragma unroll
        for (int u = 0; u < 4 * RT; u++) wide_pair<SH>(R, K, u, 0);
    }
    for (int bi = 0; bi < nblk; bi++) {
        const int b = bk0 + bi, buf = bi & 1;
        const bool more = bi + 1 < nblk;
        const uint8_t *wl = buf ? wr[1] : wr[0], *wn = buf ? wr[0] : wr[1], *xl = buf ? xr[1] : xr[0];
        wait_vm_n<NB>();
        sync();
        issue_b(b, 3);
        if (more) issue_w(b + 1, buf ^ 1);
        wide_stage<SH, 0>(wl, wn, bl, xl, R, K, kq);
        if (more) wait_vm_n<NB + NW>();
        else wait_vm_n<NB>();
        sync();
        issue_b(b, 4);
        wide_stage<SH, 1>(wl, wn, bl, xl, R, K, kq);
        if (more) wait_vm_n<NB + NW>();
        else wait_vm_n<NB>();
        sync();
        issue_b(b, 5);
        wide_stage<SH, 2>(wl, wn, bl, xl, R, K, kq);
        wait_vm_n<NB>();
        sync();
        issue_b(b, 6);
        wide_stage<SH, 3>(wl, wn, bl, xl, R, K, kq);
        wait_vm_n<NB>();
        sync();
        issue_b(b, 7);
        wide_stage<SH, 4>(wl, wn, bl, xl, R, K, kq);
        wait_vm_n<NB>();
        sync();
        if (more) issue_b(b + 1, 0);
        wide_stage<SH, 5>(wl, wn, bl, xl, R, K, kq);
        if (more) wait_vm_n<NB>();
        else wait_vm_n<0>();
        sync();
        if (more) issue_b(b + 1, 1);
        wide_stage<SH, 6>(wl, wn, bl, xl, R, K, kq);
        if (more) wait_vm_n<NB>();
        sync();
        if (more) issue_b(b + 1, 2);
        // The last block's look-ahead reads stale stage and weight bytes and drops them.
        wide_stage<SH, 7>(wl, wn, bl, xl, R, K, kq);
    }

    // The outputs to LDS (lane: row rw + 16 rt + rl of matrix m, tokens 16 g + 4
    // kq + i), then to memory in whole lines: stored straight from the MFMA
    // layout, 64 bytes a token and instruction, they took 16-20 us of a launch
    // over 256 tokens.
    wait_vm_n<0>();
    __syncthreads();
    const bool part = a.ks > 1;
    const int width = MODE == W_GLU && !part ? SH::ROWS : SH::WROWS;  // GLU partials: gate's rows, then up's
#pragma unroll
    for (int g = 0; g < TT; g++) {
        const float4 uv = *(const float4 *)&us[16 * g + 4 * kq];
        const float u4[4] = {uv.x, uv.y, uv.z, uv.w};
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int rt = 0; rt < RTM; rt++) {
                float *o = &space.out.y[16 * g + 4 * kq + i][16 * (RTM * wave + rt) + rl];
                const float v = R.acc[rt][g][i] * u4[i];
                if constexpr (MODE == W_GLU) {
                    const float up = R.acc[RTM + rt][g][i] * u4[i];
                    if (part) o[0] = v, o[SH::ROWS] = up;
                    else o[0] = glu_act(v, up, a.gelu);
                } else o[0] = v;
            }
    }
    __syncthreads();
    const int64_t ld = part ? a.nrows : a.ldy;
    const int64_t plane = (int64_t)a.M * a.nrows;
    float *out = part ? a.out + 2 * z * plane : a.out;
    const bool vec = ld % 4 == 0 && (uintptr_t)out % 16 == 0 && plane % 4 == 0 &&
                     (MODE != W_ADD || part || (uintptr_t)a.y_in % 16 == 0);
    for (int e = threadIdx.x; e < SH::TOK * width / 4; e += SH::NT) {
        const int t = e / (width / 4), c = 4 * (e % (width / 4));
        const int m = MODE == W_GLU && c >= SH::ROWS ? 1 : 0, r = row0 + c - m * SH::ROWS;
        if (t0 + t >= a.M || r >= a.nrows) continue;
        float4 v = *(const float4 *)&space.out.y[t][c];
        const int64_t o = m * plane + (t0 + t) * ld + r;
        if (vec && r + 4 <= a.nrows) {
            if (MODE == W_ADD && !part) {
                const float4 y = *(const float4 *)(a.y_in + o);
                v.x = y.x + v.x, v.y = y.y + v.y, v.z = y.z + v.z, v.w = y.w + v.w;
            }
            *(float4 *)(out + o) = v;
        } else {
            const float f[4] = {v.x, v.y, v.z, v.w};
            for (int i = 0; i < min(4, a.nrows - r); i++)
                out[o + i] = MODE == W_ADD && !part ? a.y_in[o + i] + f[i] : f[i];
        }
    }
}

// The launch of a batch of M tokens: token tiles of at most 128, evened out
// and rounded up to a built count of 16-token groups (37 tokens in a 48-token
// tile: the 13824 x 5120 gate/up 42 us, 95 us in a 128-token one); past 48
// tokens one 8-wave workgroup a CU of 256 weight rows, below it two 4-wave
// workgroups of 128, whose barriers don't hold each other up (the 14336 x 4096
// gate/up of 20 tokens 26 against 30 us, of 37 tokens 42 against 44, of 64
// tokens 41 against 40); as many splits of K (whole blocks, none empty) as
// those slots hold at once: rounded to the nearest count, the workgroups past
// the slots ran a second round (the 11008 x 4096 feed-forward block of 96 tokens 120
// us, 98 now; the 2816-wide one of 256 tokens 183, 150; the 8B's QKV of 512
// tokens as 288 workgroups on 256 CUs, its 512-token turn 20.4 ms, 19.8 now).
// The slots are an XCD's: 84 units of 3 token tiles fit the chip's 256, but four
// XCDs get 11 units, 33 workgroups on 32 CUs (the 7168 x 5120 QKV of 384 tokens in
// 3 splits 105 us, in 2 77).
struct WidePlan {
    int tt, rows, ntt, ks;
};
static WidePlan wide_plan(int64_t rows, int M, int nb, int cus, int mode) {
    WidePlan p;
    p.ntt = (M + 127) / 128;
    const int need = ((M + p.ntt - 1) / p.ntt + 15) / 16;
    p.tt = need <= 2 ? 2 : need <= 4 ? need : need <= 6 ? 6 : 8;
    p.ntt = (M + 16 * p.tt - 1) / (16 * p.tt);
    p.rows = (p.tt > 3 ? 256 : 128) / (mode == W_GLU ? 2 : 1);
    const int64_t tiles = (rows + p.rows - 1) / p.rows, slots = (p.tt > 3 ? 1 : 2) * (int64_t)cus;
    auto whole = [&](int64_t ks) {  // no split without blocks
        const int per = std::max<int>(1, (int)((nb + ks - 1) / ks));
        return std::max(1, (nb + per - 1) / per);
    };
    p.ks = whole(std::max<int64_t>(1, std::min<int64_t>({16, slots / (tiles * p.ntt), (int64_t)nb / 2})));
    while (p.ks > 1 && (tiles * p.ks + 7) / 8 * p.ntt > slots / 8) p.ks = whole(p.ks - 1);
    return p;
}
int wide_splits(int64_t rows, int M, int nb, int cus, int mode) { return wide_plan(rows, M, nb, cus, mode).ks; }

template <int MODE, int TT>
static hipError_t wide_go(WideArgs &a, const WidePlan &p, hipStream_t s) {
    using SH = WideShape<MODE, 2, TT, (TT > 3 ? 8 : 4)>;
    a.units = (a.nrows + SH::ROWS - 1) / SH::ROWS * a.ks, a.ntt = p.ntt;
    hipLaunchKernelGGL((k_gemm_wide<SH>), dim3((unsigned)(8 * a.ntt * ((a.units + 7) / 8))), dim3(SH::NT), 0, s, a);
    return hipGetLastError();
}
template <int MODE>
static hipError_t wide_mode(WideArgs &a, const WidePlan &p, hipStream_t s) {
    switch (p.tt) {
    case 2: return wide_go<MODE, 2>(a, p, s);
    case 3: return wide_go<MODE, 3>(a, p, s);
    case 4: return wide_go<MODE, 4>(a, p, s);
    case 6: return wide_go<MODE, 6>(a, p, s);
    default: return wide_go<MODE, 8>(a, p, s);
    }
}

hipError_t launch_gemm_wide(const void *w, const void *w2, int64_t ne0, int64_t ne1, const void *act, int M, int mode,
                            float *y, const float *y_in, int64_t ldy, void *scratch, int cus, hipStream_t s) {
    WideArgs a{};
    a.gelu = (mode & GLU_GELU) ? 1 : 0;
    mode &= ~GLU_GELU;
    const WidePlan p = wide_plan(ne1, M, (int)(ne0 / 256), cus, mode);
    a.w = (const uint8_t *)w, a.w2 = (const uint8_t *)w2, a.act = (const uint8_t *)act;
    a.act_stride = (int64_t)hact_bytes(ne0), a.y_in = y_in, a.ldy = ldy;
    a.nrows = (int)ne1, a.nb = (int)(ne0 / 256), a.n_in = (int)ne0, a.M = M, a.ks = p.ks;
    a.out = p.ks > 1 ? (float *)scratch : y;
    if (mode == W_GLU) return wide_mode<W_GLU>(a, p, s);
    if (mode == W_ADD) return wide_mode<W_ADD>(a, p, s);
    return wide_mode<W_STORE>(a, p, s);
}

}  // namespace ts5hip
