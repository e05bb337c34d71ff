// caps.cpp -- shape gate, backend selection, scratch planning, params packing.
//
// Counterpart of the reference's src/runtime/caps.mm:1-306. The contract is
// the same: helix_scan_supported() == false means the caller keeps its own
// kernel, selection never fails, and helix_scan_scratch_size() agrees exactly
// with what the encoder lays out. Everything here is plain C++ and runs
// without a GPU (ctx may be a host-only context or null for planning).
#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <tuple>
#include <string>
#include <vector>

#include "helix_internal.h"

namespace {

// Kernel families (helix_amd/csrc/kernels). d_state is padded to np = 64, 128
// or 256 and every family is instantiated at each np it serves.
//
//   Pass A runs the head-block kernels (pass_a_hb.hip: B split once per
//   workgroup of four items, helix_chunk_state_hb_*) up to d_state 128 and the
//   per-item kernels (pass_a_x6.hip, helix_chunk_state_x*) at d_state 256.
//   fp32 path (SGMMA, or HELIX_FORCE_BACKEND=s..., multipass, fp32 storage):
//     Pass A helix_chunk_state{_hb}_x6f32_n*  bf16x6 split products, stores
//                                        the per-chunk prefix states R_c (fp32)
//                                        and fp64 decay records
//     Pass B helix_state_scan_f32
//     Pass C helix_chunk_out_x6_n{64,128}  bf16x6 split products
//            helix_chunk_out_f32_n256      fp32 MFMA (the bf16x6 planes of a
//                                          d_state 256 tile exceed the LDS)
//   fp32 path at d_state <= 128 (fp32 storage): Pass C walks each segment's
//   chunks on bf16x6 products with the state in registers, so Pass A stores no
//   per-chunk states (HELIX_F32_WALK=0 keeps the chunk-parallel Pass C):
//     Pass A helix_chunk_state_hb_x6agg_r64_n{64,128}  segment aggregates,
//                                                      fp64 decay records
//     Pass B helix_state_scan_f32 (or the walk's prologue, fuse_b)
//     Pass C helix_scan_walk_x6_n{64,128}
//   bf16 path (AUTO or MPP, multipass): Pass C walks each segment's chunks on
//   bf16 MFMA with the state in registers; Pass A computes the segment
//   aggregates only, fp32-accurate (the reference's contract for the carried
//   state): up to d_state 128 on three products of scaled fp16 planes
//   (helix_chunk_state_hb_h3agg_{,bc_,bf16io_,f16io_}n*; HELIX_PASSA_F16=0
//   keeps six bf16 split products), otherwise on six bf16 split products, or,
//   opted into with HELIX_PASSA_SPLIT=3, on three.
//     Pass A helix_chunk_state{_hb}_x{6,3}agg_n*     fp32 storage
//            helix_chunk_state{_hb}_x{6,3}agg_bc_n*  ... also writes bf16 copies
//                                                    of B and C for the walk
//            helix_chunk_state{_hb}_x{6,3}agg_{bf16,f16}io_n*   16-bit storage
//     Pass B helix_state_scan_f32 (or the walk's prologue, fuse_b)
//     Pass C helix_scan_walk16_bf16{,_bc,_bf16io,_f16io}_n*
//   single pass (multipass = false): helix_scan_1pass_{f32,bf16io,f16io}_n*, no
//   scratch; fp32-accurate (bf16x6 products with fp32 storage up to d_state
//   128, fp32 MFMA otherwise); diagonal A: helix_scan_1pass_diag_f32_n{64,128}.

constexpr int kNps[3] = {64, 128, 256};

int np_index(int d_state) {
    if (d_state <= 64) return 0;
    if (d_state <= 128) return 1;
    return 2;
}

const char* const kIoTag[3] = {"", "bf16io_", "f16io_"};   // fp32, bf16, f16 storage

int io_index(helix_dtype io) { return io == HELIX_BF16 ? 1 : io == HELIX_F16 ? 2 : 0; }

// Traits are composed from these choices, once per process; the names live as
// long as the process.
struct TraitTable {
    // [io][k]: single pass; [k]: diagonal A; [k]: fp32 path; [k]: the fp32
    // path's walk (d_state <= 128); [io][k]: the same with 16-bit storage (io
    // 1, 2); [io][split6][bccopy][k]: bf16 path (bccopy
    // only with fp32 storage).
    HelixMatmulTraits single[3][3], diag[2], f32[3], f32walk[2], f32io[3][2], bf16[3][2][2][3], ysingle[2];
    // [io][bccopy][k]: bf16 path with Pass A on scaled fp16 planes (d_state
    // <= 128; bccopy only with fp32 storage).
    HelixMatmulTraits h3[3][2][2];
    std::vector<std::string> names;   // every kernel name, deduplicated
    std::deque<std::string> store;    // backing storage of the strings above

    const char* keep(const std::string& v) {
        store.push_back(v);
        return store.back().c_str();
    }
    const char* kernel(const std::string& v) {
        for (const std::string& n : names)
            if (n == v) return keep(v);
        names.push_back(v);
        return keep(v);
    }

    TraitTable() {
        for (int k = 0; k < 3; ++k) {
            const std::string np = std::to_string(kNps[k]);
            const std::string upto = " (d_state<=" + np + ")";
            for (int io = 0; io < 3; ++io) {
                HelixMatmulTraits& t = single[io][k];
                t = HelixMatmulTraits{};
                t.backend = HELIX_BACKEND_SGMMA;
                t.name = keep(std::string("mfma fp32, single pass") +
                              (io == 0 ? "" : io == 1 ? ", bf16 storage" : ", f16 storage") + upto);
                // fp32 storage up to d_state 128: every product on six bf16
                // split products (pass_single.hip, X6); otherwise fp32 MFMA.
                t.mfma_a = t.mfma_c = io == 0 && kNps[k] <= 128 ? "v_mfma_f32_16x16x32_bf16 (bf16x6 split operands)"
                                                                : "v_mfma_f32_16x16x4_f32";
                t.np = kNps[k];
                t.k_single = kernel(std::string("helix_scan_1pass_") + (io == 0 ? "f32_" : kIoTag[io]) + "n" + np);
                if (io == 0 && kNps[k] <= HELIX_N_BLOCK) t.k_single_acc = kernel("helix_scan_1pass_f32_acc_n" + np);
                t.single_threads = 64 * HELIX_1PASS_WAVES(kNps[k]);
            }
            if (k < 2) {
                // The single pass (fp32 storage, scalar A) run as the three
                // passes with its state tiles in y: Pass A's aggregate kernel
                // (no records), Pass B, and the fp32 path's walk forming its
                // own decay preamble.
                HelixMatmulTraits& t = ysingle[k];
                t = HelixMatmulTraits{};
                t.backend = HELIX_BACKEND_SGMMA;
                t.name = keep("mfma fp32, single pass as three launches, state tiles in y" + upto);
                t.k_chunk_state = kernel("helix_chunk_state_hb_x6agg_n" + np);
                t.k_state_scan = kernel("helix_state_scan_y_f32");
                t.k_chunk_out = kernel("helix_scan_walk_x6_y_n" + np);
                t.mfma_a = "v_mfma_f32_32x32x16_bf16 (bf16x6 split operands)";
                t.mfma_c = "v_mfma_f32_32x32x16_bf16 (bf16x6 split operands)";
                t.np = kNps[k];
                t.walk = true;
                t.walk_hb = true;
                t.a_hb = true;
            }
            if (k < 2) {
                HelixMatmulTraits& t = diag[k];
                t = HelixMatmulTraits{};
                t.backend = HELIX_BACKEND_SGMMA;
                t.name = keep("mfma fp32, single pass, diagonal A" + upto);
                t.mfma_a = t.mfma_c = "v_mfma_f32_16x16x4_f32";
                t.np = kNps[k];
                t.k_single = kernel("helix_scan_1pass_diag_f32_n" + np);
                t.single_threads = HELIX_WG;
            }
            {
                HelixMatmulTraits& t = f32[k];
                t = HelixMatmulTraits{};
                t.backend = HELIX_BACKEND_SGMMA;
                const bool x6c = kNps[k] <= 128;
                t.name = keep(std::string(x6c ? "mfma fp32, passes A and C bf16x6" : "mfma fp32, pass A bf16x6") +
                              upto);
                t.k_chunk_state = kernel(std::string(kNps[k] <= 128 ? "helix_chunk_state_hb_x6f32_n"
                                                                    : "helix_chunk_state_x6f32_n") + np);
                t.a_hb = kNps[k] <= 128;
                t.k_state_scan = kernel("helix_state_scan_f32");
                t.k_chunk_out = kernel(x6c ? "helix_chunk_out_x6_n" + np : "helix_chunk_out_f32_n" + np);
                t.mfma_a = "v_mfma_f32_32x32x16_bf16 (bf16x6 split operands)";
                t.mfma_c = x6c ? "v_mfma_f32_32x32x16_bf16 (bf16x6 split operands)" : "v_mfma_f32_32x32x2_f32";
                t.np = kNps[k];
                t.rec_kind = x6c ? 2 : 0;
            }
            if (k < 2) {
                HelixMatmulTraits& t = f32walk[k];
                t = f32[k];
                t.name = keep("mfma fp32, passes A and C bf16x6, chunk walk" + upto);
                t.k_chunk_state = kernel("helix_chunk_state_hb_x6agg_r64_n" + np);
                t.k_chunk_out = kernel("helix_scan_walk_x6_n" + np);
                t.k_chunk_out_acc = kernel("helix_scan_walk_x6_acc_n" + np);
                t.mfma_c = "v_mfma_f32_32x32x16_bf16 (bf16x6 split operands)";
                t.walk = true;
                t.walk_hb = true;
                t.walk_fuse_b = true;
                t.rec_kind = 2;
            }
            for (int io = 1; io < 3 && k < 2; ++io) {
                HelixMatmulTraits& t = f32io[io][k];
                t = f32walk[k];
                t.name = keep(std::string("mfma fp32, passes A and C bf16x6, ") + (io == 1 ? "bf16" : "f16") + " storage" + upto);
                t.k_chunk_state = kernel(std::string("helix_chunk_state_hb_x6agg_r64_") + kIoTag[io] + "n" + np);
                t.k_chunk_out = kernel(std::string("helix_scan_walk_x6_") + kIoTag[io] + "n" + np);
                t.k_chunk_out_acc = nullptr;
                t.mfma_a = io == 1 ? "v_mfma_f32_32x32x16_bf16 (one exact plane of B, three of x)"
                                   : "v_mfma_f32_32x32x16_bf16 (two exact planes of B, three of x)";
                t.mfma_c = io == 1 ? "v_mfma_f32_32x32x16_bf16 (one exact plane of B and C, three of the rest)"
                                   : "v_mfma_f32_32x32x16_bf16 (two exact planes of B and C, three of the rest)";
                t.fallback = &single[io][k];
            }
            for (int io = 0; io < 3; ++io)
                for (int s6 = 0; s6 < 2; ++s6)
                    for (int bc = 0; bc < 2; ++bc) {
                        HelixMatmulTraits& t = bf16[io][s6][bc][k];
                        t = HelixMatmulTraits{};
                        if (bc && io) continue;   // copies only from fp32 storage
                        t.backend = HELIX_BACKEND_MPP;
                        const char* split = s6 ? "x6" : "x3";
                        t.name = keep(std::string("mfma bf16 pass C, chunk walk, pass A ") +
                                      (s6 ? "bf16x6" : "bf16x3 (narrower state: opt-in)") +
                                      (io == 1 ? ", bf16 storage" : io == 2 ? ", f16 storage" : "") + upto);
                        const bool hb = kNps[k] <= 128;
                        t.k_chunk_state = kernel(std::string(hb ? "helix_chunk_state_hb_" : "helix_chunk_state_") +
                                                 split + "agg_" + (bc ? "bc_" : kIoTag[io]) + "n" + np);
                        t.a_hb = hb;
                        t.k_state_scan = kernel("helix_state_scan_f32");
                        t.k_chunk_out = kernel(std::string("helix_scan_walk16_bf16_") + (bc ? "bc_" : kIoTag[io]) +
                                               "n" + np);
                        if (io == 0 && kNps[k] <= HELIX_N_BLOCK)
                            t.k_chunk_out_acc = kernel(std::string("helix_scan_walk16_bf16_") + (bc ? "bc_" : "") +
                                                       "acc_n" + np);
                        t.bf16_state = true;
                        t.mfma_a = s6 ? "v_mfma_f32_32x32x16_bf16 (bf16x6 split operands)"
                                      : "v_mfma_f32_32x32x16_bf16 (bf16x3 split operands)";
                        t.mfma_c = hb ? "v_mfma_f32_32x32x16_bf16" : "v_mfma_f32_16x16x32_bf16";
                        t.np = kNps[k];
                        t.walk = true;
                        t.walk_hpw = HELIX_WALK16_HPW(kNps[k]);
                        t.walk_hb = hb;
                        t.walk_fuse_b = true;
                        t.bccopy = bc != 0;
                        t.rec_kind = 1;
                    }
        }
        for (int io = 0; io < 3; ++io)
            for (int k = 0; k < 2; ++k)
                for (int bc = 0; bc < 2; ++bc) {
                    HelixMatmulTraits& t = h3[io][bc][k];
                    t = bf16[io][1][bc][k];
                    if (!t.name) continue;   // copies only from fp32 storage
                    const std::string np = std::to_string(kNps[k]);
                    t.name = keep(std::string("mfma bf16 pass C, chunk walk, pass A fp16x3 (scaled planes)") +
                                  (io == 1 ? ", bf16 storage" : io == 2 ? ", f16 storage" : "") + " (d_state<=" + np + ")");
                    t.k_chunk_state = kernel(std::string("helix_chunk_state_hb_h3agg_") + (bc ? "bc_" : kIoTag[io]) + "n" + np);
                    t.mfma_a = io ? "v_mfma_f32_32x32x16_f16 (one scaled fp16 plane of B, two of x: two products)"
                                  : "v_mfma_f32_32x32x16_f16 (two scaled fp16 planes, three products)";
                }
        for (int k = 0; k < 2; ++k) h3[0][1][k].nocopy = &h3[0][0][k];
        // What helix_ctx_backend_desc reports for a descriptor run as blocks
        // of state indices on these kernels.
        auto blocks_name = [&](HelixMatmulTraits& t) {
            if (t.name) t.name_blocks = keep(std::string(t.name) + ", in blocks of at most " +
                                             std::to_string(HELIX_N_BLOCK) + " state indices");
        };
        for (auto& a : single) for (auto& t : a) blocks_name(t);
        for (auto& t : f32) blocks_name(t);
        for (auto& t : f32walk) blocks_name(t);
        for (auto& t : ysingle) blocks_name(t);
        for (auto& t : diag) blocks_name(t);
        for (auto& a : bf16) for (auto& b2 : a) for (auto& c2 : b2) for (auto& t : c2) blocks_name(t);
        for (auto& a : h3) for (auto& b2 : a) for (auto& t : b2) blocks_name(t);
    }
};

const TraitTable& table() {
    static const TraitTable t;
    return t;
}

// Pass A writes bf16 copies of B and C for the walking Pass C (fp32 storage);
// HELIX_WALK_BCCOPY=0 / 1 switches them off / on where the kernels can. At
// d_state 256 the per-item Pass A copies when the K = heads_per_group *
// n_pslab workgroups of a chunk cover its 64 rows with two quads of four state
// indices per thread (pass_a_x6.hip, copy_map). block: d is one block of
// state indices of a larger d_state.
bool bccopy_on(const helix_tuning& tu, const helix_scan_desc& d, bool block) {
    if (tu.bccopy == 0) return false;
    const long K = (long)(d.n_head / d.n_group) * ((d.head_dim + HELIX_HD - 1) / HELIX_HD);
    // The head-block Pass A (d_state <= 128) can copy at every shape (one
    // wave per 8-token block of a chunk and group, pass_a_hb.hip). The copies
    // paid off while a walk workgroup read a chunk's rows for two heads: with
    // more than eight items per group, and for blocks of state indices. The plan
    // keeps room for them there; what the encoder runs is no_copies' choice.
    if (d.d_state <= 128) return tu.bccopy == 1 || K > 8 || block;
    return (64 + K - 1) / K * (d.d_state / 4) <= 2 * 256;
}

const helix_tuning kDefaultTuning{};

const helix_tuning& tuning_of(const helix_ctx* ctx) { return ctx ? ctx->tuning : kDefaultTuning; }

// Workgroup counts the planner aims for: 256 CUs with a few resident
// workgroups each, so a launch fills the chip with a short tail.
constexpr long kTargetWgA = 512;
constexpr long kTargetWgC = 1024;

long env_long(const char* name, long dflt) {
    if (const char* v = std::getenv(name)) {
        char* end = nullptr;
        const long x = std::strtol(v, &end, 10);
        if (end != v && x > 0) return x;
    }
    return dflt;
}

int env_switch(const char* name) {   // -1 unset, else the first digit
    const char* v = std::getenv(name);
    if (!v || v[0] < '0' || v[0] > '9') return -1;
    return v[0] - '0';
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

thread_local std::string t_last_error;
thread_local const helix_ctx* t_last_ctx = nullptr;

}  // namespace

namespace helix::rt {

// Whether a short scan is faster as one launch of the single pass than as the
// passes. The single pass runs one workgroup per CU, four per (seq, head, P
// slab), each over the whole sequence: with u = rounds of 256 workgroups x
// (chunks + 1) it takes 3.7 u + 1 us (fp32 storage, d_state 65..128; 2.8 u + 1.5
// up to 64), 5.0 u + 1.5 (16-bit storage; 3.5 u + 1.5). The passes take 25-32 us
// at d_state 65..128 and 17-20 up to 64 before the length shows, the fp32 path's
// a little more than the bf16 path's. Measured at 64..640 tokens x 1..8
// sequences of 8..80 heads, 27 heads of 192: at the limits below 18-31 us
// against 18-42, one step past them 18-38 against 17-44.
namespace {
long one_launch_units(const helix_scan_desc& d) {
    const long wg = (long)d.n_seq * d.n_head * ((d.head_dim + HELIX_HD - 1) / HELIX_HD) * 4;
    return (wg + 255) / 256 * ((d.n_tok + HELIX_CS - 1) / HELIX_CS + 1);
}
}  // namespace
bool one_launch_scan(const helix_scan_desc& d, bool fp32_path) {
    const long u = one_launch_units(d);
    return u <= (d.io_dtype == HELIX_F32 ? 5 : 4) + (d.d_state > 64 ? 1 : 0) + (fp32_path ? 1 : 0);
}

helix_tuning tuning_from_env() {
    helix_tuning t;
    t.scratch_mb = env_long("HELIX_SCRATCH_MB", t.scratch_mb);
    if (const char* f = std::getenv("HELIX_FORCE_BACKEND")) t.force_fp32 = f[0] == 's' || f[0] == 'S';
    if (env_switch("HELIX_PASSA_SPLIT") == 3) t.passa_split = 3;
    t.fuse_b = env_switch("HELIX_FUSE_B");
    const int f16 = env_switch("HELIX_PASSA_F16");
    if (f16 >= 0) t.passa_f16 = f16 > 0 ? 1 : 0;
    if (t.fuse_b > 1) t.fuse_b = 1;
    const int bc = env_switch("HELIX_WALK_BCCOPY");
    t.bccopy = bc == 0 ? 0 : bc > 0 ? 1 : -1;
    t.seg_len = (int)env_long("HELIX_SEG_LEN", 0);
    t.walk_len = (int)env_long("HELIX_WALK_LEN", 0);
    t.hblk = (int)env_long("HELIX_HBLK", 0);
    t.walk_items = (int)std::min<long>(env_long("HELIX_WALK_ITEMS", 0), HELIX_HB);
    const int fw = env_switch("HELIX_F32_WALK");
    if (fw >= 0) t.f32_walk = fw > 0 ? 1 : 0;
    const int yt = env_switch("HELIX_1PASS_Y");
    if (yt >= 0) t.ytile = yt > 0 ? 1 : 0;
    const int sb = env_switch("HELIX_STATE_BLOCKS");
    if (sb >= 0) t.state_blocks = sb > 0 ? 1 : 0;
    for (const char* k : {"HELIX_PASSA_SPLIT", "HELIX_PASSA_F16", "HELIX_FUSE_B",
                          "HELIX_WALK_BCCOPY", "HELIX_SEG_LEN", "HELIX_WALK_LEN", "HELIX_WALK_ITEMS", "HELIX_HBLK", "HELIX_F32_WALK",
                          "HELIX_1PASS_Y", "HELIX_STATE_BLOCKS"})
        if (std::getenv(k)) t.planned = false;
    return t;
}

const char* const* all_kernel_names(size_t* count) {
    static const std::vector<const char*> ptrs = [] {
        std::vector<const char*> v;
        for (const std::string& n : table().names) v.push_back(n.c_str());
        return v;
    }();
    *count = ptrs.size();
    return ptrs.data();
}

void set_error(const helix_ctx* ctx, const std::string& msg) {
    t_last_ctx = ctx;
    t_last_error = msg;
}

namespace {
int choose_walk_len(const helix_scan_desc& d, int cpg);
}

namespace {
bool state_blocks_on(const helix_ctx* ctx, const helix_scan_desc& d) {
    if (d.d_state > HELIX_N_MAX) return true;   // the gate admits fp32 storage and scalar A only
    if (d.d_state <= HELIX_N_BLOCK || d.io_dtype != HELIX_F32 || d.a_form != HELIX_A_SCALAR_PER_HEAD)
        return false;
    // Measured at L=8192 H=64 P=64 G=8, d_state 160, 192 and 256: blocks of
    // 128 and less took 0.28-0.30 ms against 0.39-0.41 on the bf16 path, and
    // 0.54-0.55 against 0.71-0.72 on the fp32 path (the d_state 256 kernels
    // are the per-item Pass A and, on the fp32 path, an fp32-MFMA Pass C).
    return tuning_of(ctx).state_blocks != 0;
}
}  // namespace

int n_state_blocks(const helix_ctx* ctx, const helix_scan_desc& d) {
    if (!state_blocks_on(ctx, d)) return 1;
    const int nb0 = (d.d_state + HELIX_N_BLOCK - 1) / HELIX_N_BLOCK;
    const int base = ((d.d_state + nb0 - 1) / nb0 + 7) / 8 * 8;   // <= HELIX_N_BLOCK
    return (d.d_state + base - 1) / base;
}

helix_scan_desc state_block(const helix_ctx* ctx, const helix_scan_desc& d, int k, int* n0) {
    helix_scan_desc b = d;
    const int nb = n_state_blocks(ctx, d);
    if (nb > 1) {
        const int base = ((d.d_state + nb - 1) / nb + 7) / 8 * 8;
        b.d_state = std::min(base, d.d_state - k * base);
        if (d.d_state > HELIX_N_MAX) b.backend = HELIX_BACKEND_SGMMA;
        if (n0) *n0 = k * base;
    } else if (n0) {
        *n0 = 0;
    }
    return b;
}

helix_scan_desc plan_desc(const helix_ctx* ctx, const helix_scan_desc& d) { return state_block(ctx, d, 0, nullptr); }

const HelixMatmulTraits& select_traits(const helix_ctx* ctx, const helix_scan_desc& d) {
    // Blocks of state indices: the kernels of their blocks.
    if (n_state_blocks(ctx, d) > 1) return select_traits_unblocked(ctx, plan_desc(ctx, d), /*block=*/true);
    return select_traits_unblocked(ctx, d);
}

const HelixMatmulTraits& select_traits_unblocked(const helix_ctx* ctx, const helix_scan_desc& d, bool block) {
    const helix_tuning& tu = tuning_of(ctx);
    const TraitTable& tt = table();
    const int k = np_index(d.d_state);
    if (d.a_form == HELIX_A_DIAG_PER_CHANNEL) return tt.diag[k < 1 ? k : 1];
    const int io = io_index(d.io_dtype);
    if (!d.multipass) return tt.single[io][k];
    // HELIX_FORCE_BACKEND=s... pins the fp32 path (reference caps.mm:82-86).
    const bool bf16 = (d.backend == HELIX_BACKEND_AUTO || d.backend == HELIX_BACKEND_MPP) && !tu.force_fp32;
    if (!bf16) {
        // 16-bit storage: Pass A and the walk up to d_state 128, on B and C as
        // one (bf16) or two (f16) exact bf16 planes. At L=2048 H=64 P=64 N=128
        // G=8 in bf16 storage 54 us against 168 for the one-launch single pass
        // (HELIX_F32_WALK=0, at d_state 256, and for short scans), whose fp32
        // MFMA walks the whole sequence in each workgroup.
        if (io) return k < 2 && tu.f32_walk != 0 && !one_launch_scan(d, true) ? tt.f32io[io][k] : tt.single[io][k];
        // A walk of one chunk carries no state between chunks: where the plan
        // gives one-chunk walks (short sequences of few heads), the
        // chunk-parallel Pass C is the faster form (config 0: 23.0 against
        // 24.0 us). HELIX_F32_WALK=0 / 1 pins either form.
        const bool walk = k < 2 && (tu.f32_walk == 1 ||
                                    (tu.f32_walk < 0 && choose_walk_len(d, (d.n_tok + HELIX_CS - 1) / HELIX_CS) > 1));
        return walk ? tt.f32walk[k] : tt.f32[k];
    }
    const int bc = io == 0 && bccopy_on(tu, d, block) ? 1 : 0;
    // Pass A on two scaled fp16 planes (three products) by default up to
    // d_state 128: config 2, 0.110 against 0.117 ms on six bf16 split
    // products, s1 at the same fp32 per-element bound; HELIX_PASSA_F16=0
    // keeps the six.
    if (k < 2 && tu.passa_split != 3 && tu.passa_f16 != 0) return tt.h3[io][bc][k];
    return tt.bf16[io][tu.passa_split == 3 ? 0 : 1][bc][k];
}

// A walk workgroup reads a chunk's rows of B and C once for four items, and
// copies cost Pass A more than they save the walk: without / with them, inputs
// out of the Infinity Cache, 4096 tokens at d_state 256 158.8 / 168.7 us (8 x 1024
// tokens of 80 heads 393 / 407), 8 x 4096 tokens of 80 heads 507 / 514 and of 27
// heads of 192 509 / 514, 2 x 2000 of 48 heads in four groups 84.3 / 87.7, 8192 of
// 24 heads 83.8 / 85.5, 4 x 1000 of 8 heads of 128 38.4 / 39.5, 2 x 4096 of 64 heads
// at d_state 64 100.6 / 103.5; slower at no shape measured.
const HelixMatmulTraits& no_copies(const helix_ctx* ctx, const HelixMatmulTraits& tr) {
    return tr.nocopy && tuning_of(ctx).planned ? *tr.nocopy : tr;
}

// The form without scratch keeps its state tiles in y only where that is the
// faster form: 481 tokens of 16 heads take 79 us with tiles in y (segments must be
// long enough for a tile) and 34 in one launch, two blocks of 455 tokens x 64 heads
// x 2 sequences 155 and 136; 1824 tokens of 8 heads 95 and 101.
bool tiles_in_y_slower(const helix_ctx* ctx, const helix_scan_desc& d, const HelixMatmulTraits& tr);

const HelixMatmulTraits* short_scan_traits(const helix_ctx* ctx, const helix_scan_desc& d,
                                           const HelixMatmulTraits& tr) {
    if (!tuning_of(ctx).planned || d.a_form != HELIX_A_SCALAR_PER_HEAD || d.d_state > HELIX_N_BLOCK ||
        !(one_launch_scan(d, tr.backend == HELIX_BACKEND_SGMMA) || tiles_in_y_slower(ctx, d, tr)))
        return nullptr;
    return &table().single[io_index(d.io_dtype)][np_index(d.d_state)];
}

// The walk's prologue loads up to segs_per_group segment aggregates per
// workgroup, two at a time. Past four segments that cost more than Pass B's own
// launch in the walk of two heads per workgroup, four aggregates in flight
// (config 2, 8 segments: 149 vs 142 us; configs 4a/4b, 4 segments, fused against
// launched: 624 vs 635 and 668 vs 681 us); not measured again on the walk of
// HELIX_HB items.
constexpr int kFuseBMaxSegs = 4;

bool fuse_b_on(const helix_ctx* ctx, const HelixMatmulTraits& tr, const MultipassPlan& plan) {
    // The walk's prologue scans whole walk segments: only when they are Pass
    // A's segments too.
    if (!tr.walk_fuse_b || plan.n_groups != 1 || plan.walk_len != plan.seg_len) return false;
    const helix_tuning& tu = tuning_of(ctx);
    if (tu.fuse_b >= 0) return tu.fuse_b == 1;
    return plan.segs_per_group <= kFuseBMaxSegs;
}

namespace {

// Chunks per walk segment for a group of `cpg` chunks (the walking Pass C, which
// layout() cuts into shorter runs where it takes HELIX_HB items per workgroup;
// also Pass A's segment on the per-item kernels): enough segments that there
// are ~kTargetWgA (seq, head, P slab) items x segments, and no more (a longer
// walk keeps more of the chunk recurrence in registers and shortens Pass B), up
// to kMaxSegLen (past that the walks get too long to fill the chip: at config
// 4a, 64-chunk segments took 1.03 ms and 16-chunk ones 0.95 ms).
constexpr long kMaxSegLen = 16;
// The head-block Pass A runs one 512-thread workgroup per CU (its LDS holds
// two chunks of split B planes): ~256 workgroups fill the chip.
constexpr long kTargetWgHb = 256;

// Workgroups of HELIX_HB (head, P slab) items of a B/C group, per segment.
long item_blocks(const helix_scan_desc& d) {
    const long n_pslab = (d.head_dim + HELIX_HD - 1) / HELIX_HD;
    const long ipg = (long)(d.n_head / d.n_group) * n_pslab;
    return (long)d.n_seq * d.n_group * ((ipg + HELIX_HB - 1) / HELIX_HB);
}

int choose_walk_len(const helix_scan_desc& d, int cpg) {
    const long n_pslab = (d.head_dim + HELIX_HD - 1) / HELIX_HD;
    const long items = (long)d.n_seq * d.n_head * n_pslab;
    const long segs = std::max<long>(1, (kTargetWgA + items - 1) / items);
    const long len = std::min<long>((cpg + segs - 1) / segs, kMaxSegLen);
    return (int)std::max<long>(1, std::min<long>(len, cpg));
}

// Dispatch model of Pass A and the walk on HELIX_HB items, one workgroup per CU on
// MI355X. Workgroup b runs on XCD b % 8 (the kernels decode their logical id with
// xcd_logical_id); in each XCD, four shader engines of eight CUs take the XCD's
// workgroups round-robin, in dispatch order, and a workgroup waits for a CU of
// its own engine. Every running workgroup moves one chunk step per lat + k * load
// microseconds, load being the running workgroups over the chip (each weighted by
// the share of its items that are real); o is a fixed cost per workgroup and g
// one per segment aggregate that a walk's prologue folds in, in chunk steps.
struct DispatchCost {
    double lat, k, o, g;
};
struct PlanCost {
    DispatchCost a, c;
};
// lat, k and o fitted to each pass timed alone at up to fourteen lengths on
// thirteen shapes (600 to 8192 tokens, 1 to 8 sequences of 16 to 96 heads, some of
// several slabs), inputs out of the Infinity Cache: rms errors 4-6 % each, no
// sign of a bias in length. By kernels: d_state up to 64, up to 128.
constexpr double kFoldG = 0.1;
constexpr PlanCost kCostBf16F32[2]  = {{{2.22, 0.00354, 1.5, 0}, {4.15, 0.0101, 0.5, kFoldG}},
                                       {{2.69, 0.00426, 2.0, 0}, {4.55, 0.0114, 0.75, kFoldG}}};
constexpr PlanCost kCostBf16Io16[2] = {{{2.27, 0.00112, 1.5, 0}, {4.27, 0.00357, 0.75, kFoldG}},
                                       {{2.46, 0.00092, 3.0, 0}, {4.79, 0.00468, 1.0, kFoldG}}};
constexpr PlanCost kCostF32[2]      = {{{2.32, 0.00373, 1.5, 0}, {8.77, 0.0109, 0.25, kFoldG}},
                                       {{3.45, 0.00417, 2.0, 0}, {11.6, 0.0166, 0.25, kFoldG}}};
constexpr PlanCost kCostF32Bf16[2]  = {{{2.14, 0.00106, 1.5, 0}, {7.23, 0.00304, 0.5, kFoldG}},
                                       {{2.36, 0.00102, 3.0, 0}, {8.62, 0.00474, 0.75, kFoldG}}};
constexpr PlanCost kCostF32F16[2]   = {{{2.20, 0.0015, 1.5, 0}, {8.0, 0.0045, 0.5, kFoldG}},
                                       {{2.90, 0.00283, 2.0, 0}, {10.8, 0.00735, 0.5, kFoldG}}};
constexpr PlanCost kCostY[2]        = {{{2.29, 0.00328, 2.0, 0}, {9.04, 0.00986, 0.5, 0}},
                                       {{3.42, 0.00488, 2.0, 0}, {12.0, 0.0148, 0.5, 0}}};
constexpr int kXcds = 8, kEnginesPerXcd = 4, kCusPerEngine = 8;
constexpr long kCus = kXcds * kEnginesPerXcd * kCusPerEngine;

const PlanCost& plan_cost(const helix_scan_desc& d, const HelixMatmulTraits& tr) {
    const int n = tr.np > 64 ? 1 : 0;
    if (tr.bf16_state) return d.io_dtype == HELIX_F32 ? kCostBf16F32[n] : kCostBf16Io16[n];
    if (tr.rec_kind == 0) return kCostY[n];   // state tiles in y
    return d.io_dtype == HELIX_F32 ? kCostF32[n] : d.io_dtype == HELIX_BF16 ? kCostF32Bf16[n] : kCostF32F16[n];
}

// The workgroups of either launch over a group of cpg chunks in runs of len, of
// `items` items each, in their kernels' logical order (item block, group, run,
// sequence; or run, item block, group, sequence: walk_runs_inner).
struct PlanGrid {
    long per_run;    // item blocks x groups
    int  cpg, len, n_run, n_seq;
    double weight;   // of a run's workgroups: HELIX_HB items count 1

    PlanGrid(const helix_scan_desc& d, int cpg_, int len_, int items) : cpg(cpg_), len(len_) {
        const int ipg = d.n_head / d.n_group * ((d.head_dim + HELIX_HD - 1) / HELIX_HD);
        per_run = (long)((ipg + items - 1) / items) * d.n_group;
        n_run = (cpg + len - 1) / len;
        n_seq = d.n_seq;
        weight = (double)ipg * d.n_group / HELIX_HB;
    }
    long total() const { return per_run * n_run * n_seq; }
    int run_of(long wid, bool fold) const {
        return (int)((walk_runs_inner(fold, n_run, n_seq) ? wid : wid / per_run) % n_run);
    }
    double steps(int r, const DispatchCost& c, bool fold) const {
        return std::min(len, cpg - r * len) + c.o + (fold ? c.g * r : 0.0);
    }
    // The chunk steps of every workgroup, weighted.
    double work(const DispatchCost& c, bool fold) const {
        return weight * n_seq * (cpg + n_run * c.o + (fold ? c.g * 0.5 * n_run * (n_run - 1) : 0.0));
    }
    // No schedule is shorter than its longest workgroup, or than all of them spread evenly.
    double makespan_bound(const DispatchCost& c, bool fold) const {
        const double longest = std::max(steps(0, c, fold), steps(n_run - 1, c, fold));
        return std::max(longest, (cpg + n_run * c.o) * per_run * n_seq / kCus);
    }
};

// Makespan in chunk steps. Every running workgroup advances at the same rate, so
// each engine's queue is list-scheduled at unit speed (the order of events does
// not depend on the rate). Past 64 rounds of workgroups how the last one falls is
// a small part of the time.
double makespan(const PlanGrid& g, const DispatchCost& c, bool fold) {
    const long n = g.total();
    if (n > 64 * kCus) return g.makespan_bound(c, fold) + 0.5 * g.len;
    const long per = n / kXcds;
    double cu[kXcds * kEnginesPerXcd][kCusPerEngine] = {};
    double T = 0.0;
    for (long b = 0; b < n; ++b) {
        const long x = b % kXcds, j = b / kXcds;
        const long wid = b < per * kXcds ? x * per + j : b;
        double* e = cu[x * kEnginesPerXcd + j % kEnginesPerXcd];
        int m = 0;
        for (int i = 1; i < kCusPerEngine; ++i)
            if (e[i] < e[m]) m = i;
        e[m] += g.steps(g.run_of(wid, fold), c, fold);
        T = std::max(T, e[m]);
    }
    return T;
}

// Items per workgroup of the walk in runs of len chunks: two where that makes no
// second round of workgroups, for a chunk step then takes about 0.7 of the time on
// the fp32-accurate walk and 0.77 on the bf16 path's (a SIMD has one working wave
// instead of two), at somewhat more per workgroup. 1824 tokens of 8 heads with tiles
// in y 97 -> 78 us, 2048 of 64 heads 94 -> 79, 628 of 24 heads on the bf16 path 33
// -> 31; past one round 8192 tokens of 64 heads would go from 124 to 144. One item
// each gains no more.
int walk_items_for(const helix_scan_desc& d, int cpg, int len) {
    return PlanGrid(d, cpg, len, 2).total() <= kCus ? 2 : HELIX_HB;
}

// Microseconds of a group of cpg chunks in segments = runs of len chunks. The
// chip is busy throughout, so the integral of lat + k * load over a launch is
// lat * T + k * work. A launch of Pass B reads every segment's aggregate and
// writes every run's start state and s1; folded in, a workgroup's first chunk waits
// for s0 and the aggregates. bound: with the makespans' lower bounds instead.
double plan_us(const helix_scan_desc& d, const HelixMatmulTraits& tr, int cpg, int len, bool fold, bool bound) {
    const PlanCost& pc = plan_cost(d, tr);
    const PlanGrid g(d, cpg, len, HELIX_HB);
    const int items = walk_items_for(d, cpg, len);
    const PlanGrid gc(d, cpg, len, items);
    DispatchCost c = pc.c;
    if (items < HELIX_HB) {
        c.lat *= tr.bf16_state ? 0.77 : 0.7;
        c.o += tr.bf16_state ? 0.4 : 0.25;
    }
    const double mb = 1e-6 * d.n_seq * d.n_head * ((d.head_dim + HELIX_HD - 1) / HELIX_HD) * 64.0 * tr.np * sizeof(float);
    double us = fold ? (tr.np > 64 ? 3.0 : 0.0) : 1.0 + mb * (0.25 * g.n_run + 0.5);
    us += pc.a.k * g.work(pc.a, false) + c.k * gc.work(c, fold);
    us += pc.a.lat * (bound ? g.makespan_bound(pc.a, false) : makespan(g, pc.a, false));
    us += c.lat * (bound ? gc.makespan_bound(c, fold) : makespan(gc, c, fold));
    return us;
}

// The chunks per Pass A segment and walk run with the least modelled time, whether
// the walk folds Pass B in, and that time, over a group of cpg chunks. fold: whether
// the plan may fold. len: this length and no other (0: any). Memoized: the plan is
// remade on every encode.
//
// Against every length timed on 36 shapes of the whole range over both paths, all
// storage types and the form without scratch, the choice was within 0.3 % of the
// best on average (4 % at most). The lengths that the walk of two heads per
// workgroup had were 23 % off (4 x 1392 tokens of 64 heads of 80, bf16 storage: runs
// of 22 and 194 us against 11 and 117; 7059 tokens of 32 heads: 108 us against 68).
// Over 230 scans of 70 to 8000 tokens, most of them short, folded or not and with two
// items per workgroup or four: 0.8 % on average, 16 % at most.
struct PlanChoice {
    int len;
    double us;
    bool fold;
};
bool folds(const helix_scan_desc& d, const HelixMatmulTraits& tr, int cpg, int len) {
    // A one-chunk run on the fp32 path with fp32 storage keeps Pass B's launch:
    // the plan of a walk there has walk_len > 1.
    return tr.walk_fuse_b && (cpg + len - 1) / len <= kFuseBMaxSegs &&
           (len > 1 || tr.bf16_state || d.io_dtype != HELIX_F32);
}
PlanChoice best_plan(const helix_scan_desc& d, const HelixMatmulTraits& tr, int cpg, bool fold, int len) {
    using Key = std::tuple<const PlanCost*, int, int, int, int, int, bool, int>;
    static std::mutex mu;
    static std::map<Key, PlanChoice> memo;
    const Key key{&plan_cost(d, tr), d.n_seq, d.n_head, d.head_dim, d.n_group, cpg, fold, len};
    {
        std::lock_guard<std::mutex> lk(mu);
        const auto it = memo.find(key);
        if (it != memo.end()) return it->second;
    }
    // Lengths up to 96 chunks, and the cuts into up to sixteen, by their lower
    // bounds: few need their schedule.
    std::vector<std::tuple<double, int, bool>> cand;
    auto add = [&](int l) {
        cand.emplace_back(plan_us(d, tr, cpg, l, false, true), l, false);
        if (fold && folds(d, tr, cpg, l)) cand.emplace_back(plan_us(d, tr, cpg, l, true, true), l, true);
    };
    if (len > 0) {
        add(len);
    } else {
        for (int l = 1; l <= std::min(cpg, 96); ++l) add(l);
        for (int j = 1; j <= 16; ++j)
            if ((cpg + j - 1) / j > 96) add((cpg + j - 1) / j);
    }
    std::sort(cand.begin(), cand.end());
    PlanChoice best{0, 0.0, false};
    for (const auto& [lower, l, f] : cand) {
        if (best.len && lower >= best.us) break;
        const double t = plan_us(d, tr, cpg, l, f, false);
        if (!best.len || t < best.us) best = {l, t, f};
    }
    std::lock_guard<std::mutex> lk(mu);
    if (memo.size() > 4096) memo.clear();
    memo.emplace(key, best);
    return best;
}

// Pass A's segment (seg_len) and the walk's (walk_len, a multiple of it). On the
// kernels of HELIX_HB items segments and runs are best_plan's length; walk_len stays
// a bound of two segments or choose_walk_len's, whichever is longer, where the walk
// does not fold Pass B in (HELIX_SEG_LEN and HELIX_WALK_LEN nest runs of several
// segments). The chunk-parallel plan's Pass A takes the longest divisor of
// walk_len that still gives ~kTargetWgHb workgroups. HELIX_WALK_LEN sets walk_len,
// HELIX_SEG_LEN sets seg_len, and walk_len is then rounded to a multiple of it.
void choose_lengths(const helix_tuning& tu, const helix_scan_desc& d, const HelixMatmulTraits& tr, int cpg,
                    int* seg_len, int* walk_len) {
    int w = tu.walk_len > 0 ? std::min(tu.walk_len, cpg) : choose_walk_len(d, cpg);
    int a = w;
    if (tu.seg_len > 0) {
        a = std::min(tu.seg_len, cpg);
        w = std::max(a, (w / a) * a);
    } else if (tr.walk_hb && tu.walk_len <= 0) {
        const int n_chunks = (d.n_tok + HELIX_CS - 1) / HELIX_CS;
        const PlanChoice c = best_plan(d, tr, cpg, tu.fuse_b != 0 && cpg == n_chunks, 0);
        a = c.len;
        if (c.fold || (w == 1 && !tr.bf16_state && d.io_dtype == HELIX_F32))
            w = a;   // the second: HELIX_F32_WALK=1 where the chunk-parallel kernel is planned
        else
            w = std::max(2 * a, (w / a) * a);
    } else if (tr.a_hb) {
        const long per_seg = item_blocks(d);
        a = 1;
        for (int cand = w; cand >= 1; --cand) {
            if (w % cand) continue;
            if (per_seg * ((cpg + cand - 1) / cand) >= kTargetWgHb) {
                a = cand;
                break;
            }
        }
    }
    if (!tr.walk) w = a;
    *seg_len = a;
    *walk_len = w;
}

void layout(const helix_tuning& tu, const helix_scan_desc& d, const HelixMatmulTraits& tr, int cpg,
            MultipassPlan* pl) {
    const bool bf16_state = tr.bf16_state, walk = tr.walk, bccopy = tr.bccopy, rec = tr.rec_kind != 0;
    const int np = tr.np;
    // State scratch is stored as padded slab tiles of 64 x np (helix_params.h).
    const size_t n_pslab = (size_t)(d.head_dim + HELIX_HD - 1) / HELIX_HD;
    const size_t state = (size_t)d.n_seq * d.n_head * n_pslab * 64 * (size_t)np;
    pl->chunks_per_group = cpg;
    choose_lengths(tu, d, tr, cpg, &pl->seg_len, &pl->walk_len);
    pl->segs_per_group = (cpg + pl->seg_len - 1) / pl->seg_len;
    pl->walks_per_group = (cpg + pl->walk_len - 1) / pl->walk_len;
    pl->run_len = tr.walk_hb && tu.walk_len <= 0 ? pl->seg_len : pl->walk_len;
    pl->walk_items = tu.walk_items > 0 ? tu.walk_items : walk_items_for(d, cpg, pl->run_len);
    pl->sl_elem_bytes = bf16_state ? 2 : 4;
    pl->sl_elems = (pl->seg_len > 1 && !walk) ? state * (size_t)cpg : 0;
    pl->sg_elems = state * (size_t)pl->segs_per_group;
    pl->ld_elems = (size_t)d.n_seq * cpg * d.n_head;
    pl->sd_elems = (size_t)d.n_seq * pl->segs_per_group * d.n_head;
    pl->bc_elems = bccopy ? (size_t)d.n_seq * (size_t)cpg * HELIX_CS * d.n_group * d.d_state : 0;
    size_t off = 0;
    pl->off_sl = off; off += align256(pl->sl_elems * pl->sl_elem_bytes);
    pl->off_sg = off; off += align256(pl->sg_elems * sizeof(float));
    pl->off_ld = off; off += align256(pl->ld_elems * sizeof(float));
    pl->off_sd = off; off += align256(pl->sd_elems * sizeof(float));
    pl->off_bc = off; off += align256(pl->bc_elems * 2);
    pl->off_cc = off; off += align256(pl->bc_elems * 2);
    const size_t rec_bytes = tr.rec_kind == 1 ? HELIX_REC_WALK_BYTES : HELIX_REC64_BYTES;
    pl->rec_elems = rec ? (size_t)d.n_seq * (size_t)cpg * d.n_head * HELIX_CS * rec_bytes / sizeof(float) : 0;
    pl->off_rec = off; off += align256(pl->rec_elems * sizeof(float));
    pl->total_bytes = off;
}

}  // namespace

MultipassPlan plan_multipass(const helix_ctx* ctx, const helix_scan_desc& d, const HelixMatmulTraits& tr,
                             size_t budget_cap) {
    const helix_tuning& tu = tuning_of(ctx);
    MultipassPlan pl;
    if (d.n_tok <= 0 || d.n_seq <= 0 || d.n_head <= 0 || d.head_dim <= 0 || d.d_state <= 0 ||
        d.n_group <= 0)
        return pl;
    pl.n_chunks = (d.n_tok + HELIX_CS - 1) / HELIX_CS;

    // Default budget sized for MI355X's 288 GB: a 64-head 8K-token prefill
    // keeps all of its chunks in one group. HELIX_SCRATCH_MB=1 forces many
    // groups (reference caps.mm:170-176).
    const size_t budget = std::min((size_t)tu.scratch_mb << 20, budget_cap);
    // The most chunks per group whose layout fits the budget: all of them
    // when that fits (every BASELINE config under the default budget), else
    // a binary search (the layout grows with the chunks per group; one chunk
    // per group is the floor even past the budget).
    long lo = 1, hi = pl.n_chunks;
    auto fits = [&](long c) {
        layout(tu, d, tr, (int)c, &pl);
        return pl.total_bytes <= budget;
    };
    if (!fits(hi)) {
        while (hi - lo > 1) {
            const long mid = lo + (hi - lo) / 2;
            if (fits(mid)) lo = mid;
            else hi = mid;
        }
        layout(tu, d, tr, (int)lo, &pl);
    }
    pl.n_groups = (pl.n_chunks + pl.chunks_per_group - 1) / pl.chunks_per_group;

    // Pass C head blocks: share C.B^T over as many heads as possible while
    // keeping ~kTargetWgC workgroups per group launch.
    const int hpg = d.n_head / std::max(1, d.n_group);
    const long base = (long)d.n_seq * pl.chunks_per_group * d.n_group;
    long want_blocks = std::max<long>(1, (kTargetWgC + base - 1) / base);
    if (tu.hblk > 0) want_blocks = (hpg + tu.hblk - 1) / tu.hblk;
    want_blocks = std::min<long>(want_blocks, hpg);
    pl.hblk = (int)((hpg + want_blocks - 1) / want_blocks);
    pl.n_hblk = (hpg + pl.hblk - 1) / pl.hblk;
    return pl;
}

MultipassPlan plan_ytile(const helix_ctx* ctx, const helix_scan_desc& d, const HelixMatmulTraits& single,
                         const HelixMatmulTraits** tr_out) {
    MultipassPlan pl;
    *tr_out = nullptr;
    const helix_tuning& tu = tuning_of(ctx);
    if (tu.ytile == 0 || !single.k_single || d.a_form != HELIX_A_SCALAR_PER_HEAD || d.io_dtype != HELIX_F32 ||
        d.d_state > 128 || d.n_tok <= 0 || d.n_seq <= 0 || d.n_head <= 0 || d.head_dim <= 0 || d.n_group <= 0)
        return pl;
    // y's rows hold 16-byte tile units: channel stride 1, the others multiples
    // of four elements (the encoder also checks y's base).
    if (d.s_y[2] != 1 || (d.s_y[0] | d.s_y[1] | d.seq_y) % 4 != 0) return pl;
    const HelixMatmulTraits& tr = table().ysingle[np_index(d.d_state)];
    const long n_chunks = (d.n_tok + HELIX_CS - 1) / HELIX_CS;
    // Every segment must have the rows its tile and log-decay take, at the
    // narrowest slab width; the last segment is the shortest.
    const int n_pslab = (d.head_dim + HELIX_HD - 1) / HELIX_HD;
    const int pw_min = std::min(HELIX_HD, d.head_dim - (n_pslab - 1) * HELIX_HD);
    const long upr = pw_min / 4;
    const long rows = (16L * tr.np + 1 + upr - 1) / upr;
    auto fits = [&](long sl) {
        const long n_seg = (n_chunks + sl - 1) / sl;
        return d.n_tok - (n_seg - 1) * sl * HELIX_CS >= rows;
    };
    if (d.n_tok < rows || rows * d.s_y[0] * 4 >= (1LL << 31)) return pl;
    layout(tu, d, tr, (int)n_chunks, &pl);
    if (!fits(pl.seg_len)) {
        // Longer segments (the walk keeps its number of segments): the
        // shortest that gives every segment its rows. The whole sequence as
        // one segment always does, since n_tok >= rows.
        const int ratio = std::max(1, pl.walk_len / std::max(1, pl.seg_len));
        helix_tuning t2 = tu;
        for (long sl = std::max<long>(pl.seg_len + 1, (rows + HELIX_CS - 1) / HELIX_CS); sl <= n_chunks; ++sl) {
            if (!fits(sl)) continue;
            t2.seg_len = (int)sl;
            t2.walk_len = (int)std::min<long>(sl * ratio, n_chunks);
            break;
        }
        if (t2.seg_len <= 0) return pl = MultipassPlan{}, pl;
        layout(t2, d, tr, (int)n_chunks, &pl);
        if (!fits(pl.seg_len)) return pl = MultipassPlan{}, pl;
        if (tu.walk_len <= 0) {
            pl.run_len = pl.seg_len;
            if (tu.walk_items <= 0) pl.walk_items = walk_items_for(d, (int)n_chunks, pl.run_len);
        }
    }
    pl.n_chunks = (int)n_chunks;
    pl.n_groups = 1;
    pl.total_bytes = 0;   // nothing outside y
    pl.hblk = 1;
    pl.n_hblk = d.n_head / d.n_group;
    *tr_out = &tr;
    return pl;
}

bool tiles_in_y_slower(const helix_ctx* ctx, const helix_scan_desc& d, const HelixMatmulTraits& tr) {
    const HelixMatmulTraits* ytr = nullptr;
    if (!tr.k_single) return false;
    const MultipassPlan pl = plan_ytile(ctx, d, tr, &ytr);
    // The one launch's time as one_launch_scan has it.
    return ytr && one_launch_units(d) * (d.d_state > 64 ? 3.7 : 2.8) + 1.0 <
                      best_plan(d, *ytr, pl.n_chunks, false, pl.seg_len).us;
}

bool build_params(const helix_scan_desc& d, HelixScanParams* o, std::string* why) {
    std::memset(o, 0, sizeof(*o));
    o->n_tok = d.n_tok;
    o->n_seq = d.n_seq;
    o->n_head = d.n_head;
    o->head_dim = d.head_dim;
    o->d_state = d.d_state;
    o->n_group = d.n_group;
    o->heads_per_group = d.n_head / d.n_group;
    o->n_pslab = (d.head_dim + HELIX_HD - 1) / HELIX_HD;
    for (int i = 0; i < 3; ++i) {
        o->s_x[i] = d.s_x[i];
        o->s_b[i] = d.s_b[i];
        o->s_c[i] = d.s_c[i];
        o->s_s[i] = d.s_s[i];
        o->s_y[i] = d.s_y[i];
    }
    o->s_dt[0] = d.s_dt[0];
    o->s_dt[1] = d.s_dt[1];
    o->seq_x = d.seq_x;
    o->seq_b = d.seq_b;
    o->seq_c = d.seq_c;
    o->seq_dt = d.seq_dt;
    o->seq_s = d.seq_s;
    o->seq_y = d.seq_y;
    o->s_a = d.s_a;
    o->dt_min = d.dt_min;
    o->dt_max = d.dt_max;

    // The kernels address one chunk of a tensor through a buffer resource
    // based at the chunk's first element, with 32-bit byte offsets: every
    // stride must be non-negative and a chunk's extent stay below 2 GiB.
    const long long strides[] = {d.s_x[0], d.s_x[1], d.s_x[2], d.s_b[0], d.s_b[1], d.s_c[0],
                                 d.s_c[1], d.s_dt[0], d.s_dt[1], d.s_y[0], d.s_y[1], d.s_y[2],
                                 d.seq_x, d.seq_b, d.seq_c, d.seq_dt, d.seq_s, d.seq_y, d.s_a};
    for (long long s : strides) {
        if (s < 0) {
            if (why) *why = "negative stride";
            return false;
        }
    }
    const long long kCs = HELIX_CS - 1, kHd = HELIX_HD - 1;
    const long long spans[] = {kCs * d.s_x[0] + kHd * d.s_x[2] + 1, kCs * d.s_y[0] + kHd * d.s_y[2] + 1,
                               kCs * d.s_b[0] + d.d_state, kCs * d.s_c[0] + d.d_state,
                               kCs * d.s_dt[0] + 1};
    for (long long e : spans) {
        if (e * (long long)sizeof(float) >= (1LL << 31)) {
            if (why) *why = "one chunk of a tensor spans 2 GiB or more";
            return false;
        }
    }

    // Grid y and z are 16-bit on the hardware dispatch packet.
    const long kMaxYZ = 65535;
    const long zA = (long)d.n_seq * o->n_pslab;
    if (d.n_head > kMaxYZ || zA > kMaxYZ || d.n_seq > kMaxYZ) {
        if (why) *why = "launch grid exceeds 65535 in y or z (n_head or n_seq*n_pslab too large)";
        return false;
    }
    return true;
}

}  // namespace helix::rt

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------

extern "C" const char* helix_ctx_last_error(const helix_ctx* ctx) {
    if (!ctx) return t_last_ctx == nullptr && !t_last_error.empty() ? t_last_error.c_str() : "null context";
    return t_last_ctx == ctx ? t_last_error.c_str() : "";
}

extern "C" bool helix_scan_supported(helix_ctx* ctx, const helix_scan_desc* d) {
    if (!ctx || !d) return false;
    if (d->n_tok <= 0 || d->n_seq <= 0 || d->n_head <= 0 || d->head_dim <= 0 ||
        d->d_state <= 0 || d->n_group <= 0)
        return false;
    if (d->n_head % d->n_group != 0) return false;
    // Scalar A runs on every path; diagonal A (one decay per state index) on
    // the fp32 single-pass walk only, up to d_state 128 (an explicit bf16
    // request for it is declined, as the reference declines diagonal A).
    if (d->a_form == HELIX_A_DIAG_PER_CHANNEL) {
        if (d->d_state > 128 || d->backend == HELIX_BACKEND_MPP) return false;
    } else if (d->a_form != HELIX_A_SCALAR_PER_HEAD) {
        return false;
    }
    // Storage of x/B/C/y in F32, F16 or BF16; compute_dtype stays F32 (the
    // bf16 compute path is chosen by backend, reference caps.mm:126).
    if (d->compute_dtype != HELIX_F32) return false;
    if (d->io_dtype != HELIX_F32) {
        if (d->io_dtype != HELIX_F16 && d->io_dtype != HELIX_BF16) return false;
        // 16-bit storage with scalar A only; B and C rows are read as runs of
        // eight elements, kept 4-byte aligned by even element strides.
        if (d->a_form != HELIX_A_SCALAR_PER_HEAD) return false;
        if ((d->s_b[0] | d->s_b[1] | d->seq_b | d->s_c[0] | d->s_c[1] | d->seq_c) & 1) return false;
    }
    if (d->d_state % 8 != 0 || d->head_dim % 8 != 0) return false;
    // A larger d_state runs as blocks of state indices on the fp32 path, each
    // adding its share into y (helix::rt::state_block): fp32 storage and
    // scalar A only, and no explicit bf16 request (the reference serves its
    // bf16 Pass C at d_state 128 and 256 only, caps.mm:65-73; AUTO takes the
    // fp32 path there too, caps.mm:89-93).
    if (d->d_state > HELIX_N_MAX &&
        (d->io_dtype != HELIX_F32 || d->a_form != HELIX_A_SCALAR_PER_HEAD || d->backend == HELIX_BACKEND_MPP))
        return false;
    // B, C rows and state rows are staged as contiguous d_state vectors.
    if (d->s_b[2] != 1 || d->s_c[2] != 1 || d->s_s[2] != 1) return false;
    if (d->s_s[1] != d->d_state) return false;
    if (d->chunk != 0 && d->chunk != HELIX_CS) return false;
    // An explicit bf16 (MPP) request must be serviceable, and the bf16 Pass C
    // exists only in the multipass decomposition (reference caps.mm:66,145-147).
    if (!d->multipass && d->backend == HELIX_BACKEND_MPP) return false;
    if (d->backend == HELIX_BACKEND_REF) return false;
    HelixScanParams unused;
    return helix::rt::build_params(*d, &unused, nullptr);
}

extern "C" size_t helix_scan_scratch_size(helix_ctx* ctx, const helix_scan_desc* d) {
    // The single-pass walks (multipass = false, diagonal A, 16-bit storage off
    // the bf16 path at d_state 256) use none.
    if (!d || !d->multipass) return 0;
    const HelixMatmulTraits& tr = helix::rt::select_traits(ctx, *d);
    if (tr.k_single) return 0;
    // Blocks run one after another in the same scratch: the largest block's
    // plan. (Where y overlaps an input, up to HELIX_N_MAX, the encoder runs
    // the one-launch single pass instead, which needs none.)
    return helix::rt::plan_multipass(ctx, helix::rt::plan_desc(ctx, *d), tr).total_bytes;
}

extern "C" helix_backend helix_ctx_select_backend(helix_ctx* ctx, const helix_scan_desc* d) {
    if (!ctx || !d) return HELIX_BACKEND_REF;
    if (d->backend == HELIX_BACKEND_SGMMA) return HELIX_BACKEND_SGMMA;
    return helix::rt::select_traits(ctx, *d).backend;
}

extern "C" const char* helix_ctx_backend_desc(helix_ctx* ctx, const helix_scan_desc* d) {
    if (!ctx || !d) return "unavailable (null context)";
    if (!helix_scan_supported(ctx, d)) return "declined (shape unsupported)";
    const HelixMatmulTraits& tr = helix::rt::select_traits(ctx, *d);
    return helix::rt::n_state_blocks(ctx, *d) > 1 && tr.name_blocks ? tr.name_blocks : tr.name;
}
