// pass_c_walk_x6.hip -- Pass C as a chunk walk over four (head, P slab) items of one
// B/C group per workgroup, up to d_state 128: the fp32 path's on bf16x6 products
// (helix_scan_walk_x6_*), and the bf16 path's on single bf16 products
// (helix_scan_walk16_bf16_*; B16 below).
//
// Reference counterpart: helix_chunk_out_f32 (src/kernels/
// helix_scan_multipass.metal:225-361). One workgroup walks a run of chunks
// from its start state S_seg (Pass B) and forms every chunk's own start state R
// on the way, producing per chunk
//     y = tril(C B^T . decay) (dt x) + exp(Lcum) . (C R)        (G1, G2, G3)
//     R <- exp(L_end) R + B^T . (decay . dt . x)                  (G4)
// Every product keeps fp32 accuracy: bf16 MFMA over operands split into three
// bf16 parts (six products, fp32 accumulation), R in fp32 registers. Against
// the chunk-parallel bf16x6 Pass C (pass_c_x6.hip), whose per-chunk start
// states Pass A writes and Pass C reads back, the walk moves half the bytes.
//
// What bounds it is the sum of its matrix and vector work: under bf16 MFMA load
// the part runs at 1.8-2.0 GHz, not 2.4, and vector instructions add to the
// matrix time (44 of them for every 12 products of 32 x 32 x 16: 470 -> 600 cycles
// a wave pair, whatever their order; reordering this kernel's phases, mixing
// them by scheduling groups or giving a SIMD's two waves opposite orders
// changed nothing or cost time). So the layout does less of both per head:
//   - Wave w owns item w % 4 and its P columns 32 (w / 4) .. + 31 for all 64
//     tokens and every state index: G2, G3 and G4 run on 32 x 32 tiles, and a
//     C or B^T fragment read from LDS feeds 32 columns.
//   - B and C are split once per workgroup, for four items.
//   - x goes straight from memory into the operand layout (lane = column,
//     tokens 16 s + 8 hi + e), as in Pass A, and never touches LDS.
//   - G1 (C B^T, the same for the four items) runs on ten 16 x 16 blocks over
//     the eight waves and is shared as fp32; each wave forms its own M = C B^T
//     . decay operand in registers. The heads' M planes would not fit the LDS.
//   - The run's last chunk leaves no state (Pass B has it): no G4.
// The fp32 path's scan at L=8192 H=64 P=64 N=128 G=8 went from 237 to 199 us, at
// L=2048 from 75 to 69, at 4 x 1000 tokens of 32 heads of 128 from 128 to 109,
// against waves of 16 columns, two heads per workgroup, M planes in LDS.
//
// The bf16 path's walk (B16) is bound by memory instead: 356 MB at L=8192 H=64
// P=64 N=128 G=8 in 68 us with the inputs out of the Infinity Cache, 5.2 TB/s
// where a copy of this card reaches 4.7-5.8 (82 us with 16-column waves and two
// heads a workgroup, which staged x and its weighted copy through LDS). x loaded
// a whole chunk ahead, in registers of its own, cost 4 us there.
//
// K order: index 16 s + 8 a + 4 b + r of a group of 16 state indices (a, b in
// {0, 1}) sits at K position 8 b + 4 a + r in the C rows (perm16), so R's result
// registers (lane hi = b) are G3's operand as they stand.
//
// LDS, rows padded by 8 elements (16 consecutive operand rows start on 16
// distinct groups of four banks, and every access of the chunk loop is a
// per-lane base plus an immediate offset; an XOR swizzle spent a quarter of the
// vector instructions on addresses):
//   C    [64 t][NP n]   three bf16 planes, perm16 n order      G1, G3
//   B^T  [NP n][64 j]   three bf16 planes, natural order       G1, G4
//   CB   [64 t][64 j]   fp32, blocks on or below the diagonal  G2
// and the decay records of two chunks: 132 KiB at d_state 128, one workgroup
// per CU.
#include "helix_common.h"

// Split planes of a caller's B and C value: three bf16 parts of fp32, one of a
// bf16 value, two of an f16 value (11 significant bits: both exact).
template <typename IO> struct WX6Planes { static constexpr int value = 3; };
template <> struct WX6Planes<__bf16> { static constexpr int value = 1; };
template <> struct WX6Planes<_Float16> { static constexpr int value = 2; };

// The pair (a, b) as NPL packed bf16 parts (NPL 1 and 2: exact for values of
// that many parts).
template <int NPL>
HELIX_DEV void wx6_split(float a, float b, unsigned (&w)[NPL]) {
    if constexpr (NPL == 3)
        split3_pair(a, b, w[0], w[1], w[2]);
    else if constexpr (NPL == 2)
        split2_pair(a, b, w[0], w[1]);
    else
        w[0] = pk_bf16(a, b);
}
// Eight values as the planes of one MFMA operand.
template <int NPL>
HELIX_DEV void wx6_split8(const float (&v)[8], bf16x8 (&o)[NPL]) {
    u32x4 q[NPL];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        unsigned w[NPL];
        wx6_split<NPL>(v[2 * e], v[2 * e + 1], w);
#pragma unroll
        for (int k = 0; k < NPL; ++k) q[k][e] = w[k];
    }
#pragma unroll
    for (int k = 0; k < NPL; ++k) o[k] = __builtin_bit_cast(bf16x8, q[k]);
}

// Products of split operands a[NA] x b[NB], smallest terms first: those of the
// parts (i, j) with i + j <= 2 (six for three parts of each).
template <int NA, int NB>
HELIX_DEV f32x16 wx6_mfma(const bf16x8 (&a)[NA], const bf16x8 (&b)[NB], f32x16 acc) {
#pragma unroll
    for (int sum = 2; sum >= 0; --sum)
#pragma unroll
        for (int i = sum; i >= 0; --i)
            if (i < NA && sum - i < NB) acc = mfma_bf16(a[i], b[sum - i], acc);
    return acc;
}
template <int NA, int NB>
HELIX_DEV f32x4 wx6_mfma16(const bf16x8 (&a)[NA], const bf16x8 (&b)[NB], f32x4 acc) {
#pragma unroll
    for (int sum = 2; sum >= 0; --sum)
#pragma unroll
        for (int i = sum; i >= 0; --i)
            if (i < NA && sum - i < NB) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[sum - i], acc, 0, 0, 0);
    return acc;
}

// K position of state index i inside its group of 16: 8 a + 4 b + r -> 8 b + 4 a + r.
HELIX_DEV int wx6_perm16(int i) {
    return (i & ~12) | ((i & 4) << 1) | ((i & 8) >> 1);
}

// G1 block idx (0..9) of the lower triangle of the 4 x 4 grid of 16 x 16
// blocks: (tb, jb) = (0,0) (1,0) (1,1) (2,0) (2,1) (2,2) (3,0) ...
HELIX_DEV int wx6_tb(int idx) { return (idx >= 1) + (idx >= 3) + (idx >= 6); }
HELIX_DEV int wx6_jb(int idx) {
    const int tb = wx6_tb(idx);
    return idx - tb * (tb + 1) / 2;
}

// Lcum log2(e) as a walk keeps it: fp64, or as the bf16 path's records have it.
template <bool B16> struct WX6Lcum { typedef double type; };
template <> struct WX6Lcum<true> { typedef float type; };

constexpr int WX6_RSJ = HELIX_CS + 8;              // B^T rows (elements)
constexpr int WX6_RSM = HELIX_CS + 4;              // CB rows (floats)
template <int NP> constexpr int WX6_RSC = NP + 8;  // C rows (elements)

// A thread's C rows of a chunk: rows 8 wave + 2 (lane / 16) and the next, a run
// of NP / 16 state indices each (eight at d_state 128, half of such a run at 64).
template <int NP>
HELIX_DEV void wx6_c_run(int lane, int wave, int& j, int& n, int& pos) {
    const int c16 = lane & 15;
    const int u = NP == 128 ? c16 : (c16 & 7), hf = NP == 128 ? 0 : (c16 >> 3);
    j = 8 * wave + 2 * (lane >> 4);
    n = 8 * u + 4 * hf;
    pos = wx6_perm16(n);    // n + 4 sits 8 further
}
// Its B rows: NP / 32 consecutive tokens of four state indices, lane bits
// placed so that a load instruction reads runs of 256 bytes and 16 consecutive
// lanes write 16 distinct bank pairs of B^T.
template <int NP>
HELIX_DEV void wx6_b_rows(int lane, int wave, int& n, int& t) {
    if constexpr (NP == 128) {
        n = 64 * (wave >> 2) + 4 * ((lane & 3) | ((lane >> 4) << 2));
        t = 16 * (wave & 3) + 4 * ((lane >> 2) & 3);
    } else {
        n = 4 * (lane & 15);
        t = 8 * wave + 2 * (lane >> 4);
    }
}

// NE consecutive elements of IO at byte offset off, in storage form.
template <typename IO, int NE>
struct WX6Run {
    static constexpr int W = NE * (int)sizeof(IO) / 4;
    unsigned w[W];
    __device__ __forceinline__ void load(helix_rsrc rs, int off) {
        if constexpr (W == 2) {
            const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0);
            w[0] = v[0];
            w[1] = v[1];
        } else {
#pragma unroll
            for (int k = 0; k < W; k += 4) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, off, 4 * k, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) w[k + e] = v[e];
            }
        }
    }
    __device__ __forceinline__ float at(int e) const {
        if constexpr (sizeof(IO) == 4)
            return as_f32(w[e]);
        else
            return io_f32<IO>((unsigned short)((e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffffu)));
    }
};

// A walk's y tiles of one chunk and item (32 x 32 MFMA layout, lane (hi, lo) of
// P column pp): tile tb's register 4 r4 + r is y[t = 32 tb + 8 r4 + 4 hi +
// r][pp]. f(rsrc, byte offset, scalar byte offset, tb, register) for each; rows
// past tlen and columns past the slab width get an offset past the resource's
// range, which drops a store and reads 0; with tlen <= 0 everything is out of
// range. Where a token row of y is longer than the slab (every layout with
// channels innermost) rows past tlen are out of range by themselves and one
// offset serves every row.
template <int ES, typename Buf, typename F>
__device__ __forceinline__ void wx6_for_y(Buf* y, const HelixScanParams& p, int seq, int h, int t0, int tlen, int p0,
                                        int pw, int pp, int hi, F&& f) {
    const int sy0 = sgpr_fresh((int)p.s_y[0]), sy2 = (int)p.s_y[2];
    const unsigned bytes = tlen > 0 ? ((tlen - 1) * sy0 + (pw - 1) * sy2 + 1) * (unsigned)ES : 0u;
    const helix_rsrc ry = make_rsrc_u(y + seq * p.seq_y + h * p.s_y[1] + (long long)t0 * p.s_y[0] +
                                          (long long)p0 * p.s_y[2],
                                      bytes);
    const int voff = (4 * hi * sy0 + pp * sy2) * ES;
    if (sy0 > (pw - 1) * sy2) {
        const int v = store_off_if_lt(voff, pp, pw, 0, 1);
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int r = 0; r < 16; ++r) f(ry, v, (32 * tb + 8 * (r >> 2) + (r & 3)) * sy0 * ES, tb, r);
    } else {
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                f(ry, store_off_if_lt(voff, 32 * tb + acc_row(r, hi), tlen, pp, pw),
                  (32 * tb + 8 * (r >> 2) + (r & 3)) * sy0 * ES, tb, r);
    }
}
template <typename IO, int AUX>
__device__ __forceinline__ void wx6_store_y(const f32x16 (&acc)[2], const HelixScanParams& p,
                                               const HelixScanBuffers& b, int seq, int h, int t0, int tlen, int p0,
                                               int pw, int pp, int hi) {
    wx6_for_y<(int)sizeof(IO)>(reinterpret_cast<IO*>(b.y), p, seq, h, t0, tlen, p0, pw, pp, hi,
                             [&](helix_rsrc ry, int voff, int soff, int tb, int r) {
                                 const float v = acc[tb][r];
                                 y_store<IO, false, AUX>(ry, v, voff, soff);
                             });
}
// What y holds at the elements wx6_store_y would store (fp32 storage), 0
// where it would store nothing: for a walk that adds into y, loaded a chunk's
// work ahead of the stores.
__device__ __forceinline__ void wx6_load_y(f32x16 (&yv)[2], const HelixScanParams& p, const HelixScanBuffers& b,
                                              int seq, int h, int t0, int tlen, int p0, int pw, int pp, int hi) {
    wx6_for_y<4>(b.y, p, seq, h, t0, tlen, p0, pw, pp, hi,
               [&](helix_rsrc ry, int voff, int soff, int tb, int r) { yv[tb][r] = buf_f32(ry, voff, soff); });
}

// The start state R of a walk segment: R[nt] register 4 r4 + r = S[32 nt + 8 r4
// + 4 hi + r][p0 + 32 pt + lo], a lane's units of the state tile as they stand
// (helix_params.h). Without p.fuse_b it is Pass B's S_seg tile of the Pass A
// segment the walk segment starts at; with p.fuse_b the tiles hold Pass A's
// segment aggregates and the wave runs Pass B's recurrence here. YT: the single
// pass without scratch (HelixScanParams::ytile, never with fuse_b): the tile is
// in y.
template <int NP, bool YT>
__device__ __forceinline__ void wx6_start_state(f32x16 (&R)[NP / 32], const HelixScanParams& p,
                                                   const HelixScanBuffers& b, int seq, int h, int slab, int seg,
                                                   int p0, int pw, int pt, int lane, bool item_ok) {
    constexpr int NT = NP / 32;
    const int lo = lane & 31, hi = lane >> 5;
    const int N = p.d_state, pp = 32 * pt + lo;
    auto put = [](f32x16& t, int r4, f32x4 v) {
#pragma unroll
        for (int r = 0; r < 4; ++r) t[4 * r4 + r] = v[r];
    };
    if constexpr (YT) {
        // The tile of the walk's first Pass A segment, in y's rows of that
        // segment and the slab's columns (ytile_unit); the range covers the
        // rows the tile and its log-decay take.
        const int s = seg * (p.walk_len / p.seg_len);
        const int upr = pw >> 2;
        const unsigned rows = (unsigned)((16 * NP + 1 + upr - 1) / upr);
        const helix_rsrc ry = make_rsrc_u(b.y + ytile_base(p, seq, h, slab, s), rows * (unsigned)p.s_y[0] * 4u);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                put(R[nt], r4, __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                            ry, (int)ytile_unit(p, tile_unit(NT, pt, nt, r4, lane), pw) * 4, 0, 0)));
        return;
    }
    const float* tiles = b.s_seg + seq * p.sg_seq + state_tile_off(p, h, slab);
    auto load_tile = [&](int s, f32x16 (&T)[NT]) {
        const helix_rsrc rg = make_rsrc_u(tiles + (long long)s * p.sg_seg, 64u * NP * sizeof(float));
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) put(T[nt], r4, buf_unit<float>(rg, lane, tile_unit(NT, pt, nt, r4, 0)));
    };
    if (!p.fuse_b) {
        load_tile(seg * (p.walk_len / p.seg_len), R);
        return;
    }
    // Pass B's recurrence (helix_state_scan_f32, same operation order) up to
    // this walk's segment:
    //   carry = s0[ids[seq]];  carry = exp(segld_s) carry + D_s,  s < seg
    // The last segment's workgroup takes one more step and stores s1. Tile
    // padding (pp >= pw, n >= d_state) starts from zero, as in Pass B. ids and
    // the segment log-decays come through the scalar unit, so using them does
    // not wait for the first chunk's vector loads.
    const int src = p.has_ids ? sload_i32(b.ids, seq) : seq;
    const long long hs = (long long)h * p.s_s[0];
    const unsigned sbytes = (unsigned)(((long long)(p.head_dim - 1) * p.s_s[1] + N) * 4);
    const int soff = (int)((p0 + pp) * p.s_s[1] + 4 * hi) * 4;
    auto state_off = [&](int nt, int r4) {   // byte offset of the lane's four state values
        return store_off_if_lt(soff + 4 * (32 * nt + 8 * r4), pp, pw, 32 * nt + 8 * r4 + 4 * hi, N);
    };
    const helix_rsrc r0 = make_rsrc_u(b.s0 + src * p.seq_s + hs, b.s0 ? sbytes : 0u);   // none: reads 0
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
            put(R[nt], r4, __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r0, state_off(nt, r4), 0, 0)));
    const float* __restrict__ sd = b.segld + seq * p.sd_seq + h;
    const bool last = seg == p.n_seg - 1;
    const int nd = seg + (last ? 1 : 0);
    constexpr int BLK = 2;   // tiles in flight
    for (int sb = 0; sb < nd; sb += BLK) {
        f32x16 T[BLK][NT];
        float a[BLK];
#pragma unroll
        for (int k = 0; k < BLK; ++k) {
            const int s = min(sb + k, nd - 1);
            load_tile(s, T[k]);
            a[k] = expf(sload_f32(sd, (long long)s * p.n_head));
        }
#pragma unroll
        for (int k = 0; k < BLK; ++k) {
            if (sb + k >= nd) break;
            if (sb + k < seg) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) R[nt] = a[k] * R[nt] + T[k][nt];
            } else if (item_ok) {
                // s1[seq] = exp(segld_seg) S_seg(seg) + D_seg
                const helix_rsrc r1 = make_rsrc_u(b.s1 + seq * p.seq_s + hs, sbytes);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const f32x16 v = a[k] * R[nt] + T[k][nt];
#pragma unroll
                    for (int r4 = 0; r4 < 4; ++r4) {
                        const u32x4 w = {as_u32(v[4 * r4]), as_u32(v[4 * r4 + 1]), as_u32(v[4 * r4 + 2]),
                                         as_u32(v[4 * r4 + 3])};
                        __builtin_amdgcn_raw_buffer_store_b128(w, r1, state_off(nt, r4), 0, 0);
                    }
                }
            }
        }
    }
}

// IO: the caller's storage type of x, B, C and y.
// YT: the single pass run as the three passes without scratch
// (HelixScanParams::ytile): the start state comes from y and the decay
// preamble is formed here from dt, as Pass A forms its records (softplus, fp64
// wave scan), since there are no records.
// YACC: the walk of a block of state indices after the first (p.y_acc): y of
// each chunk is loaded with the next chunk's inputs and added to the chunk's
// result.
// B16: the bf16 path's walk: every operand rounded once to bf16, one product in
// place of six, on its Pass A's records (store_decay_record). BIO: the type B
// and C are read in; __bf16 with fp32 storage when they come from Pass A's bf16
// copies (the host points B and C there).
template <int NP, typename IO = float, bool YT = false, bool YACC = false, bool B16 = false, typename BIO = IO>
__device__ __forceinline__ void scan_walk_x6_impl(const HelixScanParams& p, const HelixScanBuffers& b) {
    static_assert(NP == 64 || NP == 128, "d_state 64 or 128");
    static_assert(sizeof(IO) == 4 || !(YT || YACC), "state tiles in y and sums into y: fp32 storage");
    constexpr int HB  = HELIX_HB;              // items per workgroup, two waves each
    constexpr int NT  = NP / 32;               // 32-row state tiles of R
    constexpr int KS  = NP / 16;               // K steps over the state (G3)
    constexpr int NPL = B16 ? 1 : WX6Planes<IO>::value;  // planes of B and C
    constexpr int NPX = B16 ? 1 : 3;           // planes of x, R and M
    static_assert(!B16 || !YT, "the form without scratch is fp32-accurate");
    static_assert(B16 || __is_same(BIO, IO), "bf16 copies of B and C: the bf16 path");
    constexpr int RSC = WX6_RSC<NP>, RSJ = WX6_RSJ, RSM = WX6_RSM;
    constexpr int PL_C = HELIX_CS * RSC, PL_B = NP * RSJ;   // one plane, elements
    constexpr int L = NP / 32;                 // B tokens per thread
    constexpr int CE = NP / 16;                // C state indices per row and thread
    __shared__ __attribute__((aligned(16))) __bf16 sC[NPL * PL_C];
    __shared__ __attribute__((aligned(16))) __bf16 sBt[NPL * PL_B];
    __shared__ __attribute__((aligned(16))) float sCB[HELIX_CS * RSM];
    // Decay records of the chunk's and the next chunk's tokens, by parity: dt
    // (0 past tlen), exp(L_end - Lcum) dt, exp(Lcum), and Lcum log2(e) in fp64
    // (B16: fp32, as its records have it): differences of Lcum keep fp32's
    // precision at any magnitude, and are exact where every Lcum is past
    // fp32's range (A at the lowest float, a state without memory).
    __shared__ __attribute__((aligned(16))) float sDt[2][HB][HELIX_CS], sW[2][HB][HELIX_CS], sE[2][HB][HELIX_CS];
    using LcumT = typename WX6Lcum<B16>::type;
    __shared__ __attribute__((aligned(16))) LcumT sL2[2][HB][HELIX_CS];

    const int lane = threadIdx.x & 63, wave = wave_uniform(), lo = lane & 31, hi = lane >> 5;
    const int N = p.d_state;

    // 1-D grid in the logical order (item block, group, walk segment,
    // sequence), as Pass A's: an XCD's share is whole token rows of one stretch
    // of a sequence, and a group's item blocks share the XCD's L2. With Pass B
    // folded in, a run reads the aggregates of all runs before it; where an XCD's
    // share is less than a sequence, the XCDs with the late runs would read them
    // all while the others have none, so from three runs on the runs of an item
    // block follow one another there instead and share an XCD (one-chunk runs over
    // four chunks, 16-bit storage: 194 tokens x 64 heads x 2 sequences 42.3 -> 33.5
    // us, 245 x 64 heads of 80 44.5 -> 32.6; 2048 x 80 heads x 2 in four runs 97.5 ->
    // 94.2; with two runs, 0.97 to 1.03 of the time either way).
    const int ipg = p.heads_per_group * p.n_pslab;
    const int ipb = p.walk_items;              // items per workgroup, at most HB
    const int nib = (ipg + ipb - 1) / ipb;
    const unsigned per_run = (unsigned)nib * (unsigned)p.n_group, per_seq = per_run * (unsigned)p.n_walk;
    const unsigned wid = xcd_logical_id(blockIdx.x, per_seq * (unsigned)p.n_seq);
    const bool runs_inner = walk_runs_inner(p.fuse_b, p.n_walk, p.n_seq);
    const unsigned inner = runs_inner ? (unsigned)p.n_walk : per_run;
    const unsigned hi_id = wid % per_seq / inner, lo_id = wid % per_seq % inner;
    const unsigned blk = runs_inner ? hi_id : lo_id;
    const int seq = (int)(wid / per_seq);
    const int seg = (int)(runs_inner ? lo_id : hi_id);
    const int ib  = (int)(blk % (unsigned)nib), g = (int)(blk / (unsigned)nib);
    // This wave's item and 32-column block of its slab. Each SIMD (waves s and
    // s + 4) holds one item; in a block of at most two items (also where the plan
    // asks for two: a grid that would leave half of the CUs idle) their four waves
    // take a SIMD each instead, and a chunk step takes about 0.8 of the time. The other waves only stage B and C and take
    // their share of G1.
    const int n_live = min(ipb, ipg - ib * ipb);
    const int is = n_live > 2 ? wave % HB : (wave % HB) >> 1;
    const int pt = n_live > 2 ? wave / HB : wave & 1;
    const bool item_ok = is < n_live && (n_live > 2 || wave < HB);
    const int ii = ib * ipb + min(is, n_live - 1);
    const int h = g * p.heads_per_group + ii / p.n_pslab;
    const int slab = ii % p.n_pslab;
    const int p0 = slab * HELIX_HD;
    const int pw = min(HELIX_HD, p.head_dim - p0);
    const int pp = 32 * pt + lo;               // this lane's column in the slab

    const int c_begin = seg * p.walk_len;
    const int c_end   = min(c_begin + p.walk_len, p.n_cg);
    if (c_begin >= c_end) return;

    constexpr int RECF = B16 ? HELIX_REC_WALK_BYTES / 4 : HELIX_REC64_BYTES / 4;   // floats per record
    const float* __restrict__ rec_h = YT ? nullptr : b.pre + ((long long)seq * p.cpg * p.n_head + h) * (HELIX_CS * RECF);
    const float* __restrict__ dt_h = b.dt + seq * p.seq_dt + h * p.s_dt[1];
    const float A_h = YT ? b.A[(long long)h * p.s_a] : 0.0f;
    const IO* __restrict__ x_h = reinterpret_cast<const IO*>(b.x) + seq * p.seq_x + h * p.s_x[1] + p0 * p.s_x[2];
    const BIO* __restrict__ B_g = reinterpret_cast<const BIO*>(b.B) + seq * p.seq_b + g * p.s_b[1];
    const BIO* __restrict__ C_g = reinterpret_cast<const BIO*>(b.C) + seq * p.seq_c + g * p.s_c[1];

    auto tlen_of = [&](int c) { return min(HELIX_CS, p.n_tok - (p.chunk_base + c) * HELIX_CS); };

    // Rows past tlen and state indices past d_state take an offset past the
    // resource's range and read 0.
    WX6Run<BIO, 4> rb[L];
    WX6Run<BIO, CE> rc[2];
    auto load_b = [&](int c, int ln) {
        constexpr int ES = (int)sizeof(BIO);
        int bn, bt;
        wx6_b_rows<NP>(ln, wave, bn, bt);
        const int tl = tlen_of(c);
        const int sb0 = sgpr_fresh((int)p.s_b[0]);
        const helix_rsrc rs = make_rsrc(B_g + (long long)(p.chunk_base + c) * HELIX_CS * p.s_b[0],
                                        ((tl - 1) * sb0 + N) * (unsigned)ES);
#pragma unroll
        for (int i = 0; i < L; ++i) rb[i].load(rs, store_off_if_lt(((bt + i) * sb0 + bn) * ES, bt + i, tl, bn, N));
    };
    auto load_c = [&](int c, int ln) {
        constexpr int ES = (int)sizeof(BIO);
        int cj, cn0, cpos;
        wx6_c_run<NP>(ln, wave, cj, cn0, cpos);
        const int tl = tlen_of(c);
        const int sc0 = sgpr_fresh((int)p.s_c[0]);
        const helix_rsrc rs = make_rsrc(C_g + (long long)(p.chunk_base + c) * HELIX_CS * p.s_c[0],
                                        ((tl - 1) * sc0 + N) * (unsigned)ES);
#pragma unroll
        for (int k = 0; k < 2; ++k) rc[k].load(rs, store_off_if_lt(((cj + k) * sc0 + cn0) * ES, cj + k, tl, cn0, N));
    };
    // K step s (tokens 16 s + 8 hi + e) of chunk c's x, in storage form. Rows
    // past tlen read 0 (past the resource's range) or, with strides under which
    // a token row is shorter than the slab, another element of the buffer, which
    // mask_x clears.
    typename IoWord<IO>::type xs[4][8];
    auto load_x = [&](int c, int s) {
        const int tl = tlen_of(c);
        const int sx0 = sgpr_fresh((int)p.s_x[0]), sx2 = (int)p.s_x[2];
        const helix_rsrc rx = make_rsrc(x_h + (long long)(p.chunk_base + c) * HELIX_CS * p.s_x[0],
                                        ((tl - 1) * sx0 + (pw - 1) * sx2 + 1) * (unsigned)sizeof(IO));
        const int xv = min(pp, pw - 1) * sx2 + 8 * hi * sx0;
#pragma unroll
        for (int e = 0; e < 8; ++e) xs[s][e] = io_load_word<IO>(rx, xv, (16 * s + e) * sx0);
    };
    // dt is 0 past tlen, but 0 times an Inf or NaN of the caller's padding is
    // not, and an MFMA spreads it over the tile's rows. Only a ragged chunk of
    // such strides comes here: a weight that ignores what it multiplies
    // (mul_legacy) would also ignore it at a token whose dt is exactly 0.
    auto mask_x = [&](int tl, int hi) {
        if (tl >= HELIX_CS || (int)p.s_x[0] > (pw - 1) * (int)p.s_x[2]) return;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (16 * s + 8 * hi + e >= tl) xs[s][e] = 0;
    };
    // The decay record of token lane (store_decay_record64: dt, exp(Lcum), Lcum
    // in fp64), or with YT the token's dt.
    u32x4 rec;
    float dtraw;
    auto load_rec = [&](int c) {
        if constexpr (YT) {
            const int tl = tlen_of(c), sdt = (int)p.s_dt[0];
            const helix_rsrc rs = make_rsrc(dt_h + (long long)(p.chunk_base + c) * HELIX_CS * p.s_dt[0],
                                            ((tl - 1) * sdt + 1) * 4u);
            dtraw = buf_f32(rs, min(lane, tl - 1) * sdt * 4, 0);
        } else {
            const helix_rsrc rs = make_rsrc(rec_h + (long long)c * p.n_head * (HELIX_CS * RECF), HELIX_CS * RECF * 4u);
            if constexpr (B16) {
                const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(rs, lane * 8, 0, 0);
                rec = u32x4{w[0], w[1], 0u, 0u};
            } else {
                rec = __builtin_amdgcn_raw_buffer_load_b128(rs, lane * 16, 0, 0);
            }
        }
    };
    // A chunk's records into buffer par, by one wave of each item.
    auto stage_rec = [&](int tl, int par) {
        if (pt != 1 || !item_ok) return;
        if constexpr (B16) {
            const float l2 = as_f32(rec[1]);
            const float l2_end = __builtin_bit_cast(float, __builtin_amdgcn_readlane((int)rec[1], 63));
            sDt[par][is][lane] = as_f32(rec[0]);
            sW[par][is][lane] = __builtin_amdgcn_exp2f(l2_end - l2) * as_f32(rec[0]);
            sE[par][is][lane] = __builtin_amdgcn_exp2f(l2);
            sL2[par][is][lane] = l2;
            return;
        }
        float dtv, e;
        double lcum;
        if constexpr (YT) {
            // As Pass A's hb_preamble forms the records.
            dtv = keep_if_lt(helix_dt(p, dtraw), lane, tl);
            lcum = wave_incl_sum((double)A_h * (double)dtv);
            e = expf((float)lcum);
        } else {
            dtv = as_f32(rec[0]);
            e = as_f32(rec[1]);
            lcum = __builtin_bit_cast(double, (unsigned long long)rec[2] | ((unsigned long long)rec[3] << 32));
        }
        sDt[par][is][lane] = dtv;
        sW[par][is][lane] = exp2_diff(bcast(lcum, 63), lcum) * dtv;
        sE[par][is][lane] = e;
        sL2[par][is][lane] = lcum * 1.4426950408889634074;
    };
    auto stage_c = [&](int ln) {
        int cj, cn0, cpos;
        wx6_c_run<NP>(ln, wave, cj, cn0, cpos);
        __bf16* const wC = sC + cj * RSC + cpos;
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int m = 0; m < CE / 4; ++m) {   // four state indices at K position cpos + 8 m
                unsigned w[2][NPL];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    if constexpr (__is_same(BIO, __bf16))
                        w[e][0] = rc[k].w[2 * m + e];   // bf16 pairs as they are
                    else
                        wx6_split<NPL>(rc[k].at(4 * m + 2 * e), rc[k].at(4 * m + 2 * e + 1), w[e]);
                }
#pragma unroll
                for (int pl = 0; pl < NPL; ++pl)
                    *reinterpret_cast<u32x2*>(wC + pl * PL_C + k * RSC + 8 * m) = u32x2{w[0][pl], w[1][pl]};
            }
    };
    // B's planes as B^T wants them: tokens bt .. bt + L - 1 of state index bn + k.
    auto stage_b = [&](int ln) {
        int bn, bt;
        wx6_b_rows<NP>(ln, wave, bn, bt);
        __bf16* const wB = sBt + bn * RSJ + bt;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            unsigned w[L / 2][NPL];
#pragma unroll
            for (int i = 0; i < L / 2; ++i) {
                if constexpr (__is_same(BIO, __bf16))   // the halves k % 2 of the two tokens' words as one pair
                    w[i][0] = __builtin_amdgcn_perm(rb[2 * i + 1].w[k >> 1], rb[2 * i].w[k >> 1],
                                                    (k & 1) ? 0x07060302u : 0x05040100u);
                else
                    wx6_split<NPL>(rb[2 * i].at(k), rb[2 * i + 1].at(k), w[i]);
            }
#pragma unroll
            for (int pl = 0; pl < NPL; ++pl) {
                __bf16* dst = wB + pl * PL_B + k * RSJ;
                if constexpr (L == 4)
                    *reinterpret_cast<u32x2*>(dst) = u32x2{w[0][pl], w[1][pl]};
                else
                    *reinterpret_cast<unsigned*>(dst) = w[0][pl];
            }
        }
    };

    load_c(c_begin, lane);
    load_b(c_begin, lane);
    load_rec(c_begin);

    // The segment's start state, R[nt] register 4 r4 + r = S[32 nt + 8 r4 + 4 hi
    // + r][pp]: a lane's units of the state tile as they stand (helix_params.h).
    f32x16 R[NT];
    wx6_start_state<NP, YT>(R, p, b, seq, h, slab, seg, p0, pw, pt, lane, item_ok);
    if constexpr (YT) {
        // The start state lies in y's rows that this workgroup's waves
        // overwrite from the first chunk on: every wave has it in registers
        // before the first barrier, which comes before any y store.
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float v = R[nt][r];
                asm volatile("" ::"v"(v));
            }
    }
    stage_c(lane);
    stage_rec(tlen_of(c_begin), 0);
    // x is first used after the chunk's second barrier.
#pragma unroll
    for (int s = 0; s < 4; ++s) load_x(c_begin, s);
    load_c(min(c_begin + 1, c_end - 1), lane);
    load_rec(min(c_begin + 1, c_end - 1));

    // Three barriers per chunk: (1) the chunk's planes and records are staged;
    // (2) CB is written and G1 and G3 are done with C (the next chunk's C
    // planes and records are staged behind it); (3) G4 is done with B^T, G2
    // with CB (the next chunk's B^T planes are written at the top of the loop).
#pragma unroll 1
    for (int c = c_begin; c < c_end; ++c) {
        const int t0   = (p.chunk_base + c) * HELIX_CS;
        const int tlen = tlen_of(c);
        const int par  = (c - c_begin) & 1;
        // The segment's last chunk leaves no state (Pass B has it): no G4, and
        // nothing staged or loaded for a next one.
        const bool last = c + 1 == c_end;
        const int cnn = min(c + 2, c_end - 1);

        // Lane-derived addresses are formed anew in every chunk: hoisted out of
        // the loop they would not fit the registers, and a spilled address is
        // reloaded behind the loads in flight.
        const int ln = vgpr_fresh(lane);
        const int lo = ln & 31, hi = ln >> 5, c16 = ln & 15, q = ln >> 4;

        stage_b(ln);
        if (!last) load_b(c + 1, ln);
        __syncthreads();   // (1)
        f32x16 yprev[2];
        if constexpr (YACC) wx6_load_y(yprev, p, b, seq, h, t0, item_ok ? tlen : 0, p0, pw, pp, hi);

        const __bf16* const rC16 = sC + c16 * RSC + 8 * q;    // operand row c16 of C
        const __bf16* const rBt = sBt + (16 * (q >> 1) + 4 * (q & 1) + (c16 >> 2)) * RSJ + 4 * (c16 & 3);

        // ---- G1: D[j][t] = (B C^T) of blocks idx = wave, wave + 8 -----------
        // Block idx: D[j = 16 jb + 4 q + r][t = 16 tb + c16].
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int idx = wave + 8 * i;
            if (idx < 10) {
                const int tb = wx6_tb(idx), jb = wx6_jb(idx);
                const __bf16* const ra = rBt + 16 * jb;
                const __bf16* const rcb = rC16 + 16 * tb * RSC;
                f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int s = 0; s < NP / 32; ++s) {
                    // B rows j = 16 jb + c16 by transpose reads of B^T: K slot
                    // 4 a + r of lane group q is C's position 32 s + 8 q + 4 a
                    // + r, state index 32 s + 16 (q / 2) + 8 a + 4 (q % 2) + r
                    // (perm16); lane 4 r + v names that row of B^T and tokens
                    // 16 jb + 4 v .. + 3.
                    bf16x8 av[NPL], bv[NPL];
#pragma unroll
                    for (int pl = 0; pl < NPL; ++pl) {
                        const u32x2 a0 = lds_read_tr16(ra + pl * PL_B + 32 * s * RSJ);
                        const u32x2 a1 = lds_read_tr16(ra + pl * PL_B + (32 * s + 8) * RSJ);
                        av[pl] = __builtin_bit_cast(bf16x8, u32x4{a0[0], a0[1], a1[0], a1[1]});
                        bv[pl] = *reinterpret_cast<const bf16x8*>(rcb + pl * PL_C + 32 * s);
                    }
                    d = wx6_mfma16(av, bv, d);
                }
                *reinterpret_cast<f32x4*>(&sCB[(16 * tb + c16) * RSM + 16 * jb + 4 * q]) = d;
            }
        }

        // ---- G3: y = exp(Lcum_t) . (C R), R the state before this chunk -----
        const __bf16* const rC = sC + lo * RSC + 8 * hi;      // operand row lo of C
        f32x16 acc[2];
        acc[0] = zero16();
        acc[1] = zero16();
        if (item_ok) {
            auto split_r = [&](int s, bf16x8 (&rp)[NPX]) {
                float rv[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) rv[e] = R[s >> 1][8 * (s & 1) + e];
                wx6_split8<NPX>(rv, rp);
            };
            auto read_c = [&](int s, bf16x8 (&cv)[2][NPL]) {
#pragma unroll
                for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                    for (int pl = 0; pl < NPL; ++pl)
                        cv[tb][pl] = *reinterpret_cast<const bf16x8*>(rC + pl * PL_C + 32 * tb * RSC + 16 * s);
            };
            bf16x8 cv[2][2][NPL], rp[2][NPX];
            read_c(0, cv[0]);
            split_r(0, rp[0]);
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                if (s + 1 < KS) {
                    read_c(s + 1, cv[(s + 1) & 1]);
                    split_r(s + 1, rp[(s + 1) & 1]);
                }
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) acc[tb] = wx6_mfma(cv[s & 1][tb], rp[s & 1], acc[tb]);
            }
#pragma unroll
            for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    const f32x4 e4 = *reinterpret_cast<const f32x4*>(&sE[par][is][32 * tb + 8 * r4 + 4 * hi]);
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[tb][4 * r4 + r] *= e4[r];
                }
        }
        __syncthreads();   // (2)

        // ---- G2: y += M . dtX, K step by K step of 16 tokens ----------------
        const float* const rCB = sCB + lo * RSM + 8 * hi;     // row lo of a tile of CB
        const __bf16* const rB = sBt + lo * RSJ + 8 * hi;     // operand row lo of B^T
        auto g2 = [&] {
            LcumT lt[2];
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) lt[tb] = sL2[par][is][32 * tb + lo];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                float v[8];
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    const f32x4 d4 = *reinterpret_cast<const f32x4*>(&sDt[par][is][16 * s + 8 * hi + 4 * a]);
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[4 * a + k] = d4[k] * io_widen<IO>(xs[s][4 * a + k]);
                }
                bf16x8 x2[NPX];
                wx6_split8<NPX>(v, x2);
                // M[t][j] = CB[t][j] exp(Lcum_t - Lcum_j), j <= t, of t tile tb
                // at tokens j = 16 s + 8 hi + e.
                const int lim = vgpr_fresh(lo - 8 * hi);
#pragma unroll
                for (int tb = s >> 1; tb < 2; ++tb) {
                    float m[8];
#pragma unroll
                    for (int a = 0; a < 2; ++a) {
                        const f32x4 cb = *reinterpret_cast<const f32x4*>(rCB + 32 * tb * RSM + 16 * s + 4 * a);
                        LcumT lj[4];
                        __builtin_memcpy(lj, __builtin_assume_aligned(&sL2[par][is][16 * s + 8 * hi + 4 * a], 16),
                                         sizeof(lj));
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const int e = 4 * a + k;
                            const float d = cb[k] * __builtin_amdgcn_exp2f((float)(lt[tb] - lj[k]));
                            m[e] = (s >> 1) == tb ? (lim >= 16 * (s & 1) + e ? d : 0.0f) : d;
                        }
                    }
                    bf16x8 mp[NPX];
                    wx6_split8<NPX>(m, mp);
                    acc[tb] = wx6_mfma(mp, x2, acc[tb]);
                }
            }
        };
        // ---- G4: R <- exp(L_end) R + B^T . (w x), w = exp(L_end - Lcum) dt ---
        auto g4 = [&] {
            const float a_c = sE[par][is][HELIX_CS - 1];   // exp(L_end)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) R[nt] *= a_c;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                float v[8];
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    const f32x4 w4 = *reinterpret_cast<const f32x4*>(&sW[par][is][16 * s + 8 * hi + 4 * a]);
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[4 * a + k] = w4[k] * io_widen<IO>(xs[s][4 * a + k]);
                }
                bf16x8 x4[NPX];
                wx6_split8<NPX>(v, x4);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    bf16x8 bp[NPL];
#pragma unroll
                    for (int pl = 0; pl < NPL; ++pl)
                        bp[pl] = *reinterpret_cast<const bf16x8*>(rB + pl * PL_B + 32 * nt * RSJ + 16 * s);
                    R[nt] = wx6_mfma(bp, x4, R[nt]);
                }
            }
        };
        if (!last) {
            __builtin_amdgcn_sched_barrier(0);
            stage_c(ln);
            load_c(cnn, ln);
            stage_rec(tlen_of(c + 1), par ^ 1);
            load_rec(cnn);
            __builtin_amdgcn_sched_barrier(0);
        } else {
            mask_x(tlen, hi);   // only a sequence's last chunk is ragged
        }
        if (item_ok) g2();
        if (!last && item_ok) {
            g4();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < 4; ++s) load_x(c + 1, s);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (YACC) {
            acc[0] += yprev[0];
            acc[1] += yprev[1];
        }
        // Reading Pass A's bf16 copies: nt alone (HELIX_NT_L2).
        constexpr int YAUX = sizeof(IO) == 4 && __is_same(BIO, __bf16) ? HELIX_NT_L2 : HELIX_NT;
        if (item_ok) wx6_store_y<IO, YAUX>(acc, p, b, seq, h, t0, tlen, p0, pw, pp, hi);
        if (last) break;
        __syncthreads();   // (3)
    }
}

#define HELIX_PASS_C_WALK_X6(NP)                                                                 \
    extern "C" __global__ __launch_bounds__(HELIX_HB_THREADS) void helix_scan_walk_x6_n##NP(   \
        HelixScanParams p, HelixScanBuffers b) {                                                \
        scan_walk_x6_impl<NP>(p, b);                                                             \
    }                                                                                           \
    extern "C" __global__ __launch_bounds__(HELIX_HB_THREADS) void helix_scan_walk_x6_bf16io_n##NP( \
        HelixScanParams p, HelixScanBuffers b) {                                                \
        scan_walk_x6_impl<NP, __bf16>(p, b);                                                        \
    }                                                                                           \
    extern "C" __global__ __launch_bounds__(HELIX_HB_THREADS) void helix_scan_walk_x6_f16io_n##NP( \
        HelixScanParams p, HelixScanBuffers b) {                                                \
        scan_walk_x6_impl<NP, _Float16>(p, b);                                                      \
    }                                                                                           \
    /* The single pass without scratch (HelixScanParams::ytile). */                             \
    extern "C" __global__ __launch_bounds__(HELIX_HB_THREADS) void helix_scan_walk_x6_y_n##NP( \
        HelixScanParams p, HelixScanBuffers b) {                                                \
        scan_walk_x6_impl<NP, float, true>(p, b);                                                \
    }                                                                                           \
    /* The walks of the second and later blocks of state indices. */                            \
    extern "C" __global__ __launch_bounds__(HELIX_HB_THREADS) void helix_scan_walk_x6_acc_n##NP( \
        HelixScanParams p, HelixScanBuffers b) {                                                \
        scan_walk_x6_impl<NP, float, false, true>(p, b);                                         \
    }

HELIX_PASS_C_WALK_X6(64)
HELIX_PASS_C_WALK_X6(128)

// The bf16 path's walk.
#define HELIX_PASS_C_WALK_BF16(NAME, NP, ...)                                                   \
    extern "C" __global__ __launch_bounds__(HELIX_HB_THREADS) void helix_scan_walk16_bf16_##NAME##n##NP( \
        HelixScanParams p, HelixScanBuffers b) {                                                \
        scan_walk_x6_impl<NP, __VA_ARGS__>(p, b);                                               \
    }
#define HELIX_PASS_C_WALK_BF16_ALL(NP)                                                          \
    HELIX_PASS_C_WALK_BF16(, NP, float, false, false, true)                                     \
    HELIX_PASS_C_WALK_BF16(bc_, NP, float, false, false, true, __bf16)                          \
    HELIX_PASS_C_WALK_BF16(bf16io_, NP, __bf16, false, false, true)                             \
    HELIX_PASS_C_WALK_BF16(f16io_, NP, _Float16, false, false, true)                            \
    /* The second and later blocks of state indices. */                                         \
    HELIX_PASS_C_WALK_BF16(acc_, NP, float, false, true, true)                                  \
    HELIX_PASS_C_WALK_BF16(bc_acc_, NP, float, false, true, true, __bf16)

HELIX_PASS_C_WALK_BF16_ALL(64)
HELIX_PASS_C_WALK_BF16_ALL(128)
