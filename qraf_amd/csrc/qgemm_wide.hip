// qgemm_wide.hip -- batched Q8_0 / Q4_0 GEMM on the 32x32x16 matrix products,
// for tile-major weights and batches over 16 rows.
//
// Same product, operand planes and error bound as qgemm.hip: per quant block
// the matrix cores accumulate sum_k q (x_hi + x_lo) in fp32, then one FMA per
// output applies the block's scale.
//
// A workgroup owns 32 TM batch rows x 64 WN weight rows.  Its waves are WN wide
// along the weight rows and WK deep along K: K group g takes every WK-th pair of
// quant blocks, and the groups' sums meet once, in LDS, at the end, so small
// products fill the chip without partial slices in memory.  A pair (64 elements
// of K) is the stage of the LDS ring: X rows then come in 128-byte pieces
// (64-byte ones reached 28 bytes per clock and CU from L2, 128-byte ones 50).
// Direct-to-LDS loads fill NS stages of X, shared by the WN waves of a group, and
// WS of the wave's own weights; one barrier per pair (none for WN = 1).
//
// 32x32x16 products and not 16x16x32: an X fragment read from LDS serves twice the
// outputs (registers only, 8 independent accumulators: 2,247 TFLOP/s against 1,183).
// What bounds the loop is the vector ALU beside them: per unit of four products (a
// 32 x 32 tile of one block, 128 matrix cycles) 16 scale FMAs, 18 (TM 2) or 9 (TM 4)
// of the weights' conversion, which overlap the products only in part.  An iteration
// of 4 / 8 / 16 units takes 0.8-0.9 / 1.1-1.4 / 1.6-1.75 us at TM 1 / 2 / 4, that is 25 /
// 31-39 / 49-53% of the matrix rate; over the whole launch (MI355X, Q4_0 11008 x 2048 at
// 128 rows, 24.2 us) the products take 30% of the waves' cycles, the VALU issues in
// 42% (in two fifths of the products' cycles) and 31% wait for LDS, memory or the
// barrier.  Against the forms of qgemm.hip (MI355X, GEMM and partial sums, Q4_0):
// 11008 x 2048 at 32 / 64 / 128 rows 14.2 / 21.9 / 30.1 -> 10.8 / 14.4 / 23.2 us, 2560 x 2048
// at 128 rows 16.0 -> 10.3, 2048 x 11008 at 128 / 512 rows 26.7 / 63.2 -> 23.7 / 54.2; Q8_0
// 2048 x 11008 at 203 rows 52.1 -> 33.6.
#include <type_traits>

#include "common.h"
#include "qgemm.h"

namespace qraf_hip {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// One lane's 8 consecutive quants as the bf16 and the fp16 MFMA operand.
// Q4_0 (one word, nibble i = element i): byte j is copied under the exponent of
// 1024 twice (v_perm), so the low half reads 1024 + e(2j) and the high half
// 1024 + 16 e(2j+1); one packed fp16 FMA takes both to e - 8, exactly.  Those
// integers have at most two mantissa bits, so the high byte of each fp16 is the
// same number as a bf8 (E5M2), which the packed bf8 conversion widens to bf16.
__device__ __forceinline__ void widen_q4(uint32_t q, uint32_t magic, u32x4& bf, u32x4& hf) {
    const f16x2 mul = {(_Float16)1.0f, (_Float16)0.0625f}, off = {(_Float16)-1032.0f, (_Float16)-72.0f};
    uint32_t h[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        constexpr uint32_t sel[4] = {0x04000400u, 0x04010401u, 0x04020402u, 0x04030403u};
        const uint32_t t = __builtin_amdgcn_perm(magic, q, sel[j]) & 0xFFF0FF0Fu;
        h[j] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, t), mul, off));
        hf[j] = h[j];
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t b = __builtin_amdgcn_perm(h[2 * j + 1], h[2 * j], 0x07050301u);
        bf[2 * j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(b, 1.0f, false));
        bf[2 * j + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(b, 1.0f, true));
    }
}
__device__ __forceinline__ void widen_q8(uint32_t a, uint32_t b, u32x4& bf, u32x4& hf) {
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t d = j ? b : a;
        const float f0 = (float)(int8_t)(d), f1 = (float)(int8_t)(d >> 8);
        const float f2 = (float)(int8_t)(d >> 16), f3 = (float)(int8_t)(d >> 24);
        bf[2 * j] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f1), __builtin_bit_cast(uint32_t, f0), 0x07060302u);
        bf[2 * j + 1] =
            __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, f3), __builtin_bit_cast(uint32_t, f2), 0x07060302u);
        hf[2 * j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(f0, f1));
        hf[2 * j + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(f2, f3));
    }
}

// The lane number, computed where it is used (not kept in a register over a loop)
__device__ __forceinline__ uint32_t lane_here() {
    uint32_t l;
    __asm__ volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}
// dma16 with the LDS byte address as a number
__device__ __forceinline__ void dma16s(v4i rsrc, uint32_t voff, uint32_t lds, int at) {  // at: a constant
    __asm__ volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds"
                     :
                     : "v"(voff), "s"(rsrc), "s"(lds), "i"(at)
                     : "memory", "m0", "scc");
}

template <int FMT, int TM, int TN, int WN, int WK, int NS, int WS>
struct WideGeom {
    static constexpr int TB = FMT == 8 ? 576 : 288;  // bytes of a 16-row tile's block
    static constexpr int NWV = WN * WK, MT = 32 * TM, NT = 32 * TN * WN;
    static constexpr int XI = 8 * TM, XW = XI / WN;     // X instructions per stage: of a K group, of a wave
    static constexpr int XG = XW / 2;                   // row groups of a wave
    static constexpr int XSTAGE = XI * 1024;
    static constexpr int WPT = 2 * TB / 16;             // 16-byte pieces of a 16-row tile's two blocks
    static constexpr int WIT = (WPT + 63) / 64, WI = 2 * TN * WIT;  // W instructions: per such tile, per stage of a wave
    static constexpr int WSLOT = 2 * TN * 2 * TB;
    static constexpr int LDS_X = WK * NS * XSTAGE, LDS_W = NWV * WS * WSLOT;
    // loads younger than the next stage's when it is waited for: an iteration issues
    // W of stage it + WS, then X of stage it + NS - 1
    static constexpr int YOUNG = (NS - 2) * (XW + WI);
    static_assert(WS == NS - 1, "weights as far ahead as X");
    static constexpr int RED = NWV * TM * TN * 4096;  // the SwiGLU epilogue: every wave's sums
    static constexpr int GIVE = WK == 2 ? TM * TN / 2 : TM * TN;  // tiles a wave hands to the other K groups
    static_assert(WK > 1 && NWV * GIVE * 4096 <= RED, "epilogue");
    static constexpr int LDS = LDS_X + LDS_W > RED ? LDS_X + LDS_W : RED;
    static_assert(LDS <= 160 * 1024, "LDS");
    static_assert(XI % WN == 0, "X split");
    static constexpr int MINB = LDS <= 80 * 1024 && NWV <= 4 ? 2 : 1;
};

template <int FMT, int TM, int TN, int WN, int WK, int NS, int WS>
__global__ __launch_bounds__(64 * WN * WK, (WideGeom<FMT, TM, TN, WN, WK, NS, WS>::MINB)) void qgemm_wide_kernel(
    const uint8_t* __restrict__ Wt, int N, int nb, const uint16_t* __restrict__ xh, const uint16_t* __restrict__ xl,
    int K, int M, int bps, int ntiles, int mchunks, int S, float* Y, const float* add, size_t slice,
    uint16_t* __restrict__ act_hi, uint16_t* __restrict__ act_lo) {
    using G = WideGeom<FMT, TM, TN, WN, WK, NS, WS>;
    constexpr int TB = G::TB, U = TM * TN;
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN, g = wave / WN;
    const int l32 = lane & 31, half = lane >> 5;

    // workgroup -> (tile, split, batch chunk): consecutive ids go to the XCDs in
    // turn, so each XCD takes a contiguous run of (split, tile, chunk): the chunks of
    // a weight tile share its L2, and so do the tiles of a split its X columns
    const int total = ntiles * mchunks * S, per = (total + 7) >> 3;
    const int lin = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || lin >= total) return;
    auto uni = [](int v) { return __builtin_amdgcn_readfirstlane(v); };  // divisions run on the VALU
    const int mc = uni(lin % mchunks), tile = uni((lin / mchunks) % ntiles), split = uni(lin / (mchunks * ntiles));
    const int m0 = mc * G::MT, n0 = tile * G::NT + wn * 32 * TN;
    const int b_begin = split * bps, b_end = min(nb, b_begin + bps);  // bps even
    const int npair = (b_end - b_begin + 1) >> 1;                    // pairs of quant blocks
    static_assert((WK & (WK - 1)) == 0 && TN == 2, "shape");
    const int nit = (npair + WK - 1) / WK;  // the same for every group: the last pair of some may not exist

    const int ntile16 = (N + 15) / 16;
    const uint32_t xb = (uint32_t)(min(M - m0, G::MT) * (K * 2));
    const v4i xrh = make_rsrc_words((const uint8_t*)xh + (size_t)m0 * K * 2, xb);
    const v4i xrl = make_rsrc_words((const uint8_t*)xl + (size_t)m0 * K * 2, xb);
    const int t16 = min(n0 >> 4, ntile16 - 1);
    const v4i wrs = make_rsrc_words(Wt + (size_t)t16 * nb * TB, (uint32_t)(min(ntile16 - t16, 2 * TN) * nb * TB));

    // X: one instruction moves rows 8 r .. +7 (r: row group) of a plane, the 128 bytes
    // of a pair each; the slot of a row's 16-byte piece is piece ^ ((row >> 1) & 7),
    // so the 16 rows of an LDS read phase fall on all 64 banks.  A wave takes row
    // groups of one parity.  Rows past M lie past the resource's end (read as
    // nothing; their outputs are not stored).
    static_assert(WN <= 2, "row groups of one parity, or of both");
    const int par = wn;  // WN == 1: both, the odd ones' pieces ^ 4
    auto xpiece = [&](uint32_t l) { return (l & 7) ^ (4u * par + (l >> 4)); };
    const uint32_t xlane = (uint32_t)((lane >> 3) * (K * 2)) + (xpiece(lane) << 4);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)lds;
    const uint32_t xbase = lds0 + (uint32_t)g * NS * G::XSTAGE, wbase = lds0 + G::LDS_X + (uint32_t)wave * WS * G::WSLOT;
    auto with = [](v4i r, uint32_t records) {
        r[2] = __builtin_amdgcn_readfirstlane((int)records);
        return r;
    };
    // X and weights of this group's pair of iteration `it`; past the group's pairs
    // nothing is in range, and of a last half pair only the first block
    uint32_t xsrc = 0, xodd = 0, xrec = 0;
    auto aim_x = [&](int it) {
        const int p = g + WK * it;
        xrec = p < npair ? xb : 0u;
        xsrc = xlane + (uint32_t)(b_begin + 2 * p) * 64u;
        if (WN == 1) xodd = xsrc + (xpiece(lane_here()) & 4 ? -64u : 64u);
        if (b_begin + 2 * p + 1 >= b_end) {
            const uint32_t past = xpiece(lane_here()) >> 2 << 31;
            if (WN == 1) xodd |= past ^ 0x80000000u;
            xsrc |= past;
        }
    };
    // this wave's q-th row group of the stage, both planes
    auto issue_x = [&](int q, int buf) {
        const uint32_t at = xbase + (uint32_t)(buf * G::XSTAGE + wn * 2048);
        const int r = q * WN + wn;
        const uint32_t v = (WN == 1 && (q & 1) ? xodd : xsrc) + (uint32_t)(r * 8 * (K * 2));
        dma16s(with(xrh, xrec), v, at, q * WN * 2048);
        dma16s(with(xrl, xrec), v, at, q * WN * 2048 + 1024);
    };
    auto issue_w = [&](int it, int slot) {
        const int p = g + WK * it;
        const uint32_t rec = p < npair ? (uint32_t)wrs[2] : 0u, l = lane_here();
#pragma unroll
        for (int q = 0; q < 2 * TN; q++) {  // 16-row tile q of the wave
            const uint32_t o = (uint32_t)((min(q, ntile16 - 1 - t16) * nb + b_begin + 2 * p) * TB);
#pragma unroll
            for (int i = 0; i < G::WIT; i++)
                if (l < (uint32_t)(G::WPT - i * 64))
                    dma16s(with(wrs, rec), l * 16 + o + i * 1024u,
                           wbase + (uint32_t)(slot * G::WSLOT), q * 2 * TB + i * 1024);
        }
    };

    float acc[TM][TN][16];
    f32x16 d[2];
#pragma unroll
    for (int t = 0; t < TM; t++)
#pragma unroll
        for (int u = 0; u < TN; u++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[t][u][r] = 0.f;
    d[0] = d[1] = f32x16{};
    float sP = 0.f;

    // X fragment of a tile: row l32, piece 4 j + 2 half + s; the plane at +1024 of each 8 rows
    const uint32_t xrow = (uint32_t)((l32 >> 3) * 2048 + (l32 & 7) * 128 + (((2 * half) ^ (l32 >> 1 & 7)) << 4));
    const int wrow = (l32 >> 4) * 2 * TB;  // the lane's 16-row tile
    const int rr = l32 & 15;
    const uint8_t* wrd = lds + G::LDS_X + (size_t)wave * WS * G::WSLOT + wrow;

    struct Raw {
        uint32_t s;
        uint32_t q[FMT == 8 ? 4 : 2];
    };
    auto read_w = [&](Raw (&r)[2][TN], int slot, int it) {
        const int left = b_end - b_begin - 2 * (g + WK * it);  // blocks from this pair on
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int u = 0; u < TN; u++) {
                const uint8_t* p = wrd + slot * G::WSLOT + u * 4 * TB + j * TB;
                if constexpr (FMT == 8) {
                    r[j][u].s = *(const uint32_t*)(p + 4 * rr);
                    const u32x4 v = *(const u32x4*)(p + 64 + 32 * rr + 16 * half);
#pragma unroll
                    for (int i = 0; i < 4; i++) r[j][u].q[i] = v[i];
                } else {
                    r[j][u].s = *(const uint16_t*)(p + 2 * rr);
                    const uint2 v = *(const uint2*)(p + 32 + 16 * rr + 8 * half);
                    r[j][u].q[0] = v.x;
                    r[j][u].q[1] = v.y;
                }
                r[j][u].s = j < left ? r[j][u].s : 0u;  // a block past the end adds nothing
            }
    };
    // one plane's fragments of a 32-row batch tile: both k steps
    struct Frag {
        u32x4 v[2];
    };
    Frag fh, fl;
    // at: xrow in the stage's buffer, toggled for the block and the k step
    auto read_x = [&](Frag& f, uint32_t at, int t, int plane) {
        f.v[0] = *(const u32x4*)(lds + at + t * 8192 + plane * 1024);
        f.v[1] = *(const u32x4*)(lds + (at ^ 16u) + t * 8192 + plane * 1024);
    };
    u32x4 wf[2][2], wh[2][2];
    uint32_t magic = 0x64646464u;
    __asm__("" : "+v"(magic));  // in a VGPR: v_perm takes one scalar operand, its selector
    float sc[2] = {0.f, 0.f};
    auto widen = [&](const Raw& r, int u) {
        if constexpr (FMT == 8) {
            sc[u] = __builtin_bit_cast(float, r.s);
            widen_q8(r.q[0], r.q[1], wf[u][0], wh[u][0]);
            widen_q8(r.q[2], r.q[3], wf[u][1], wh[u][1]);
        } else {
            sc[u] = (float)__builtin_bit_cast(_Float16, (uint16_t)r.s);
            widen_q4(r.q[0], magic, wf[u][0], wh[u][0]);
            widen_q4(r.q[1], magic, wf[u][1], wh[u][1]);
        }
    };
    Raw raw[2][2];
    auto hi = [&](const Frag& f, int u, int s, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, f.v[s]),
                                                      __builtin_bit_cast(bf16x8, wf[u][s]), c, 0, 0, 0);
    };
    auto lo = [&](int u, int s, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, fl.v[s]),
                                                     __builtin_bit_cast(f16x8, wh[u][s]), c, 0, 0, 0);
    };
    // the scale FMAs of a finished product (tile t, columns u)
    auto apply = [&](int t, int u, const f32x16& v, float s) {
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][u][r] = __builtin_fmaf(v[r], s, acc[t][u][r]);
    };
    // A pair's 2 TM tiles.  The pipeline runs across tiles, blocks and pairs: at a
    // tile's first unit its fragments and the first columns' weights are in (or on
    // their way to) registers; the FMAs of a unit issue among the next unit's MFMAs.
    // land(): called when every X fragment of the pair has been read, before the
    // last tile's units: it makes the next stage's data readable.
    auto pair_units = [&](uint32_t at, uint32_t nat, auto&& issue, auto&& land) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
#pragma unroll
            for (int t = 0; t < TM; t++) {
                const bool last = t == TM - 1, end = last && j == 1;
                const int nt = last ? 0 : t + 1;
                const uint32_t xat = end ? nat : at ^ (j || last ? 64u : 0u);
                const float sp = t == 0 ? sP : sc[1];
                if (t == 0) widen(raw[j][1], 1);
                if (end) land();
                d[0] = hi(fh, 0, 0, f32x16{});
                d[0] = hi(fh, 0, 1, d[0]);
                d[0] = lo(0, 0, d[0]);
                d[0] = lo(0, 1, d[0]);
                apply(t == 0 ? TM - 1 : t - 1, 1, d[1], sp);
                __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (j == 0) issue(2 * t);
                __builtin_amdgcn_sched_barrier(0);
                const float s0 = sc[0];
                d[1] = hi(fh, 1, 0, f32x16{});
                d[1] = hi(fh, 1, 1, d[1]);
                __builtin_amdgcn_sched_barrier(0);
                read_x(fh, xat, nt, 0);
                d[1] = lo(1, 0, d[1]);
                d[1] = lo(1, 1, d[1]);
                apply(t, 0, d[0], s0);
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
                __builtin_amdgcn_sched_barrier(0);
                read_x(fl, xat, nt, 1);
                if (last) widen(raw[end ? 0 : 1][0], 0);
                __builtin_amdgcn_sched_barrier(0);
                if (j == 0) issue(2 * t + 1);
                __builtin_amdgcn_sched_barrier(0);
                sP = sc[1];
            }
        }
    };
#pragma unroll
    for (int s = 0; s < NS - 1; s++) {
        aim_x(s);
#pragma unroll
        for (int q = 0; q < G::XG; q++) issue_x(q, s);
        issue_w(s, s);
    }
    int xbuf = 0, wslot = 0, xnext = NS - 1;
    // stage 0
    wait_vm_lgkm0<G::YOUNG>();
    if constexpr (WN > 1) lds_barrier();
    read_w(raw, 0, 0);
    const uint32_t xat0 = (uint32_t)(g * NS * G::XSTAGE) + xrow;
    read_x(fh, xat0, 0, 0);
    read_x(fl, xat0, 0, 1);
    widen(raw[0][0], 0);
    for (int it = 0; it < nit; it++) {
        const int nbuf = xbuf + 1 == NS ? 0 : xbuf + 1, nslot = wslot + 1 >= WS ? 0 : wslot + 1;
        aim_x(it + NS - 1);
        pair_units(xat0 + (uint32_t)(xbuf * G::XSTAGE), xat0 + (uint32_t)(nbuf * G::XSTAGE), [&](int k) {
            // spread over the units: a burst would hold the wave at the load queue,
            // and with it the matrix cores
            if (k == 0) {
                __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | (0 << 8));  // the raw weights are in registers
                issue_w(it + WS, wslot);
            }
            constexpr int PER = (G::XG + U - 1) / U;
#pragma unroll
            for (int i = 0; i < PER; i++)
                if (k * PER + i < G::XG) issue_x(k * PER + i, xnext);
        }, [&]() {
            // the next stage has landed (later ones may be in flight), this one's X has been read by every wave
            wait_vm_lgkm0<G::YOUNG>();
            if constexpr (WN > 1) lds_barrier();
            read_w(raw, nslot, it + 1);
        });
        xbuf = nbuf;
        wslot = nslot;
        xnext = xnext + 1 == NS ? 0 : xnext + 1;
    }
    wait_vm_lgkm0<0>();
    apply(TM - 1, 1, d[1], sP);

    // ---- epilogue.  The K groups' sums meet in LDS and are added in group order.
    f32x4* red = (f32x4*)lds;
    if (!act_hi) {
        // tile q is finished by group q % WK and stored straight from registers:
        // bounds by the resource (rows) and the lane's offset (columns), so a store
        // is an add and the store itself
        lds_barrier();
#pragma unroll
        for (int q = 0; q < U; q++)
            if (q % WK != g)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float* a = acc[q / TN][q % TN] + 4 * i;
                    red[((wave * G::GIVE + (WK == 2 ? q >> 1 : q)) * 4 + i) * 64 + lane] = f32x4{a[0], a[1], a[2], a[3]};
                }
        __syncthreads();
        const uint32_t rec = (uint32_t)(min(M - m0, G::MT) * N) * 4u;
        const rsrc_t yr = make_rsrc(Y + (size_t)split * slice + (size_t)m0 * N, rec);
        const rsrc_t ar = make_rsrc(add + (size_t)m0 * N, rec);
        const uint32_t rowb = (uint32_t)N * 4u;
#pragma unroll
        for (int q = 0; q < U; q++) {
            if (q % WK != g) continue;
            float(&a)[16] = acc[q / TN][q % TN];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const f32x4 own = f32x4{a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3]};
                f32x4 v = own;
#pragma unroll
                for (int k = 0; k < WK; k++) {
                    const f32x4 p = k == q % WK ? own : red[(((k * WN + wn) * G::GIVE + (WK == 2 ? q >> 1 : q)) * 4 + i) * 64 + lane];
                    v = k ? v + p : p;
                }
#pragma unroll
                for (int r = 0; r < 4; r++) a[4 * i + r] = v[r];
            }
            const int n = n0 + 32 * (q % TN) + l32;
            const uint32_t at = n < N ? (uint32_t)n * 4u + (uint32_t)(4 * half) * rowb : 0x80000000u;
            if (add) {
                float av[16];
#pragma unroll
                for (int r = 0; r < 16; r++)
                    av[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                          ar, at + (uint32_t)(32 * (q / TN) + 8 * (r >> 2) + (r & 3)) * rowb, 0, 0));
#pragma unroll
                for (int r = 0; r < 16; r++) a[r] += av[r];
            }
#pragma unroll
            for (int r = 0; r < 16; r++)
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, a[r]), yr,
                                                      at + (uint32_t)(32 * (q / TN) + 8 * (r >> 2) + (r & 3)) * rowb, 0, 0);
        }
        return;
    }
    // SwiGLU: every wave's sums through LDS, then a loop over units of 4 rows of one
    // column (tile (t, u) of wave column w, rows 8 i + 4 half .. + 3)
    const int F2 = N >> 1;
    constexpr int UNITS = WN * U * 4;  // of 64 lanes
    lds_barrier();                     // the stages are no longer read
#pragma unroll
    for (int q = 0; q < U; q++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float* a = acc[q / TN][q % TN] + 4 * i;
            red[((wave * U + q) * 4 + i) * 64 + lane] = f32x4{a[0], a[1], a[2], a[3]};
        }
    __syncthreads();
#pragma unroll 2
    for (int j = wave; j < UNITS; j += G::NWV) {
        const int w = j / (U * 4), q = (j >> 2) % U, i = j & 3;
        f32x4 v = red[j * 64 + lane];
#pragma unroll
        for (int k = 1; k < WK; k++) v += red[(k * UNITS + j) * 64 + lane];
        const int n = tile * G::NT + w * 32 * TN + 32 * (q % TN) + l32;
        const int m = m0 + 32 * (q / TN) + 8 * i + 4 * half;
        // gate and up columns in neighbouring lanes: the even lane takes rows 0 and 2, the odd lane 1 and 3
        const bool odd = lane & 1;
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
            const float give = odd ? v[r] : v[r + 1], got = __shfl_xor(give, 1);
            const float gate = odd ? got : v[r], up = odd ? v[r + 1] : got;
            const int mm = m + r + (odd ? 1 : 0);
            if (mm < M && n < N) {
                const size_t e = (size_t)mm * F2 + (n >> 1);
                split_bf16(silu_gate(gate, up), &act_hi[e], &act_lo[e]);
            }
        }
    }
}

// ------------------------------------------------------------------ launch

template <int FMT, int TM, int TN, int WN, int WK, int NS, int WS>
static int wide_attr() {
    QH_CHECK_HIP(hipFuncSetAttribute((const void*)qgemm_wide_kernel<FMT, TM, TN, WN, WK, NS, WS>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)WideGeom<FMT, TM, TN, WN, WK, NS, WS>::LDS));
    return QRAF_HIP_OK;
}

// forms: index, TM, WN, WK, then NS, WS for Q4_0 and for Q8_0
#define QW_FORMS(X) \
    X(0, 4, 2, 2, 2, 1, 2, 1) X(1, 2, 2, 2, 2, 1, 2, 1) X(2, 2, 1, 4, 2, 1, 2, 1) X(3, 1, 1, 4, 3, 2, 3, 2)
#define QW_T(i, TM, WN, WK, N4, W4, N8, W8) {32 * TM, 64 * WN, WK},
static constexpr QwTile QW_TILE[] = {QW_FORMS(QW_T)};
static_assert(sizeof(QW_TILE) / sizeof(QW_TILE[0]) == QW_FORM_COUNT, "forms");
QwTile qgemm_wide_tile(int form) { return QW_TILE[form]; }

int qgemm_wide_init() {
#define QW_A(i, TM, WN, WK, N4, W4, N8, W8)           \
    QH_TRY((wide_attr<4, TM, 2, WN, WK, N4, W4>()));  \
    QH_TRY((wide_attr<8, TM, 2, WN, WK, N8, W8>()));
    QW_FORMS(QW_A)
#undef QW_A
    return QRAF_HIP_OK;
}
template <int FMT, int TM, int WN, int WK, int NS, int WS>
static void wide_go(int grid, hipStream_t s, const void* Wt, int N, int K, const uint16_t* xh, const uint16_t* xl, int M,
                    int bps, int nt, int mch, int S, float* Y, const float* add, size_t slice, uint16_t* act_hi,
                    uint16_t* act_lo) {
    hipLaunchKernelGGL((qgemm_wide_kernel<FMT, TM, 2, WN, WK, NS, WS>), dim3(grid), dim3(64 * WN * WK),
                       (WideGeom<FMT, TM, 2, WN, WK, NS, WS>::LDS), s, (const uint8_t*)Wt, N, K / 32, xh, xl, K, M, bps,
                       nt, mch, S, Y, add, slice, act_hi, act_lo);
}

int launch_qgemm_wide(int form, const void* Wt, uint32_t dtype, int N, int K, const uint16_t* xh, const uint16_t* xl,
                      int M, float* Y, const float* add, int S, int bps, uint16_t* act_hi, uint16_t* act_lo,
                      hipStream_t s) {
    const QwTile t = QW_TILE[form];
    const int nt = (N + t.nt - 1) / t.nt, mch = (M + t.mt - 1) / t.mt;
    const long long total = (long long)nt * mch * S;
    QH_REQUIRE(total < (1LL << 30), QRAF_HIP_ERR_INVALID, "qgemm: batch %d too large", M);
    const int grid = (int)((total + 7) / 8 * 8);
    const size_t slice = S > 1 ? (size_t)M * N : 0;
#define QW_L(i, TM, WN, WK, N4, W4, N8, W8)                                                                            \
    case i:                                                                                                             \
        if (dtype == DT_Q8_0)                                                                                           \
            wide_go<8, TM, WN, WK, N8, W8>(grid, s, Wt, N, K, xh, xl, M, bps, nt, mch, S, Y, add, slice, act_hi, act_lo); \
        else                                                                                                            \
            wide_go<4, TM, WN, WK, N4, W4>(grid, s, Wt, N, K, xh, xl, M, bps, nt, mch, S, Y, add, slice, act_hi, act_lo); \
        break;
    switch (form) { QW_FORMS(QW_L) }
#undef QW_L
    QH_CHECK_HIP(hipGetLastError());
    return QRAF_HIP_OK;
}

}  // namespace qraf_hip
