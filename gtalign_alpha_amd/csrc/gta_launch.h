// gta_launch.h -- host-side launchers of the stage kernels (gta_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <algorithm>
#include "gta_device.h"

namespace gta {

enum { DPM_IBEST_L = 0, DPM_GRAND_L = 1, DPM_CONSTRAINED_L = 2 };
enum { RM_DPREFINE_L = 0, RM_FIN1_L = 1, RM_FIN2_L = 2, RM_PROD1_L = 3, RM_PROD2_L = 4, RM_FIN2F_L = 5,
       RM_PROD2F_L = 6, RM_PROD2L_L = 7 };

struct DpLaunch {
    int mode;          // DPM_*_L
    int gap0;
    float gapopen;
    int usess;         // cell score: 0 distance, 1 distance + SS bonus, 2 SS match + residue similarity
    float ssw;
    int dpscan;
    float rrw;         // residue-score weight of kind 2
};

// Pairs of a chunk split by the form of their DP fill.
struct DpBuckets {
    const int* small;                       // one wave per pair (nullptr: every pair)
    int nsmall;
    // one workgroup of W = 4 << g waves per pair, g = 0, 1, 2
    const int* mw[3];
    int nmw[3];
    int* failflag;     // set by a W-wave or grid fill whose row wait gave up
    // pairs whose strips are spread over one-wave workgroups (dp_grid_items)
    const int* grid;
    int ngrid;
    const int* gstrip0;                     // [ngrid + 1] first strip item of each pair
    int* gnext;                             // the item counter, then [ngrid] strips done
    float* grows;                           // per pair nstrips x Lr floats at growoff[k]
    const unsigned long long* growoff;
    size_t growtot;                         // floats of all grid pairs' rows
    int gworkers;                           // one-wave workgroups that take strips
    // any pair outside the one-wave list
    bool any_big() const { return nmw[0] > 0 || nmw[1] > 0 || nmw[2] > 0 || ngrid > 0; }
};

// Pairs of a chunk split by refinement size: `small` pairs (nullptr: every
// pair) take one workgroup each; each `big` pair's slots are split over
// several workgroups whose part records (partbuf, nbig x parts entries) are
// merged by a second kernel.
struct RefSplit {
    const int* small;
    int nsmall;
    const int* big;
    int nbig;
    int seeds_per_part;    // seed diagonals per workgroup in the seed search
    int slots_per_part;    // fragment slots per workgroup in the refinements
    void* partbuf;
};

// Workgroups of a refinement launch over the DP alignments.
struct RefineShape {
    int waves;         // per workgroup of unsplit pairs
    int wgs;           // workgroups of a persistent grid: 16 waves per CU
    int ldscap;        // alignments up to this length are staged in LDS
    int split_waves;   // the same of split pairs' workgroups
    int split_ldscap;
};

// Waves per workgroup of the DPRefine launches over a chunk of `pairs` pairs
// whose alignments have up to `maxaln` positions.  A launch ends with its longest
// alignments, whose slots (about 6 per 40 positions) wait for each other in the
// workgroup's 8 slot groups a wave, so larger workgroups make it shorter until
// the device is full of them; then smaller ones leave fewer lanes idle while a
// pair's last slots run.  The longer the longest alignment is beside the others,
// the more pairs it takes to hide it: the lines follow maxaln.  28 launches with
// 1, 2 and 4 waves, ms:
//   up to 90 positions: 1,000 pairs 3.0, 2.0, 2.0; 4,500 2.9, 2.6, 2.9; 10,000 3.9,
//     3.7, 4.2; 16,000 4.6, 4.7, 5.7; 64,000 9.2, 14.1, 22.3
//   up to 140: 12,800 pairs 13.3, 11.1, 12.5; 44,000 27.3, 27.9, 38.0
//   up to 200: 4,000 pairs 12.2, 7.7, 6.1; 16,000 14.4, 13.2, 18.0; 40,000 20.5,
//     22.1, 34.7; 64,000 37, 44, 71
//   up to 300: 15,000 pairs 18.1, 12.4, 12.1; 54,000 45.6, 43.9, 53.6; 79,000
//     45.0, 49.9, 80.8
//   up to 1,000: 4 x 1,500 24.7, 15.1, 11.3; 16,000 pairs 128, 56, 43; 64,000 153,
//     128, 156; 16 x 12,000 176, 174, 216; 16 x 50,000 661, 712, 888
// One-wave workgroups also stage only alignments of up to rlds_cap32(1)
// positions in LDS; longer ones are read from L2 in every pass, so one wave is
// used when at most 15% of the pairs can have longer ones (fits1; 16 x 50,000: 7%;
// 1 x 500,000: 27%, 0.40 s with two waves and 0.50 with one).
// The at most 8 slots of up to 47 positions fit one wave: 99 pairs 0.69, 0.74,
// 0.76; 16,000 2.1, 2.8, 3.2; 64,000 5.4, 9.3, 11.8.  In a small batched chunk the
// 4,096 one-wave workgroups of the persistent grid would take longer to find
// the queue empty: 54 pairs 2.5, 2.0, 1.8; 10,000 3.7, 3.4, 3.1; 30,000 8.0, 8.7,
// 8.4.
inline int dprefine_waves(int ncu, long long pairs, int maxaln, bool fits1, bool batched) {
    const double percu = (double)pairs / ncu;
    if (maxaln <= 47) return batched && percu <= 64.0 ? 4 : 1;
    if (percu <= std::min(64.0, 4.0 + maxaln / 5.0)) return 4;
    return percu <= std::min(1024.0, 0.9 * maxaln) || !fits1 ? 2 : 1;
}

// Waves per workgroup of the final stage's launches over `live` pairs (0: not
// known, as in the batched form).  Few pairs reach it, whose second phases run
// 128 slots: 64 slot groups take them in two rounds.  Where the pairs keep every
// CU busy, half as many groups leave fewer of them idle and let a second
// workgroup work while one waits; the longer the longest alignment, the later.
// 4 launches with 8 and 4 waves, ms (longest alignment, pairs per CU):
//   FP32: 211, 1.6 0.26, 0.24; 221, 4.0 0.90, 1.13; 334, 5.8 1.19, 1.48; 400, 5.9
//     0.99, 1.10; 400, 11.7 1.67, 1.53; 546, 13 2.95, 2.75; 78, 6.7 0.56, 0.54; 100,
//     15.6 1.30, 0.91
//   FP64, of which a CU holds 8 waves: 100, 1.0 0.20, 0.20; 211, 3.5 0.77, 0.56;
//     400, 2.3 0.84, 0.81; 400, 3.5 1.10, 0.96; 568, 4.1 2.03, 2.97; 900, 2.3 2.13, 2.50;
//     221, 23 7.3, 5.3
inline int final_waves(int prec, int ncu, long long live, int maxaln) {
    const double percu = (double)live / ncu;
    return percu <= (prec ? std::max(1.0, maxaln / 130.0) : std::max(2.0, maxaln / 50.0)) ? FINAL_WAVES
                                                                                         : FINAL_WAVES / 2;
}

// The shape of the launch of refinement `mode` over `pairs` pairs of alignments
// of up to `maxaln` positions (the final stage's: the live pairs, 0 where the
// host does not know them).  The log search's steps run in order in one slot
// group, so its pairs take workgroups of REFINE_WAVES; the FULLA searches, of
// 768 slots a pair, workgroups of FINAL_WAVES; split pairs, each many
// workgroups, take at most REFINE_WAVES.  The FP32 forms stage in LDS what leaves
// room for 16 waves per CU at their own workgroup size (1 x 200 pairs of 2,900
// residues, split: with the unsplit pairs' LDS 102 ms of DPRefine, with their own
// 68); the FP64 ones, which run 8, up to 1,536 positions.
inline RefineShape refine_shape(int prec, int mode, int ncu, long long pairs, int maxaln, bool fits1,
                                bool batched) {
    RefineShape s;
    s.waves = mode == RM_DPREFINE_L ? dprefine_waves(ncu, pairs, maxaln, fits1, batched)
              : mode == RM_PROD2L_L ? REFINE_WAVES
              : mode == RM_FIN2F_L || mode == RM_PROD2F_L ? FINAL_WAVES
                                                          : final_waves(prec, ncu, pairs, maxaln);
    s.wgs = ncu * 16 / s.waves;
    s.split_waves = std::min(s.waves, REFINE_WAVES);
    s.ldscap = s.split_ldscap = std::min(maxaln, 1536);
    if (prec == 0 || mode == RM_DPREFINE_L) {
        s.ldscap = std::min(s.ldscap, rlds_cap32(s.waves));
        s.split_ldscap = std::min(s.split_ldscap, rlds_cap32(s.split_waves));
    }
    return s;
}

struct RefineLaunch {
    int dinv;
    int epi, dpi, maxndpiters;
    float prescore;
    RefineShape shape;
};

hipError_t launch_secstr(const DevChunk& C, hipStream_t st);
hipError_t launch_init(const DevChunk& Q, const DevChunk& R, const DevState& S, hipStream_t st);
// the pair score d02 / (d02 + d2) over device arrays of n operands
hipError_t launch_pair_score(const float* d02, const float* d2, int n, float* out, hipStream_t st);
// the solve's square root (kind 0), reciprocal (1) or division (2) over the same
hipError_t launch_solve_op(int kind, const float* a, const float* b, int n, float* out, hipStream_t st);
// the VALU calibration kernel of instruction kind `kind` (0-7) on the first
// `lanes` lanes of every wave
hipError_t launch_valu_calib(float* out, int blocks, int iters, int kind, int lanes, hipStream_t st);
// the reference filter after the stage-1 prescreen, per block of qgroup queries (0: all)
hipError_t launch_keep_refs(const DevChunk& Q, const DevChunk& R, const DevState& S, int qgroup,
                            hipStream_t st);
// the superposition searches run in the reference's FP32 arithmetic in both
// precision forms (their result is a choice of superposition, which the final
// stage refines in the precision of the form)
hipError_t launch_findfrag(const DevChunk& Q, const DevChunk& R, const DevState& S,
                           const Geom& G, int dinv, const RefSplit& Sp, hipStream_t st);
hipError_t launch_refine_gapless(const DevChunk& Q, const DevChunk& R, const DevState& S,
                                 const Geom& G, int dinv, const RefSplit& Sp, hipStream_t st);
// per-length d0/d8 tables on the current device (once per device, before any launch)
hipError_t upload_length_tables();
// wq.items != nullptr: a persistent grid of pgrid workgroups drains the
// work queue instead of the small bucket (batched form)
hipError_t launch_dp(const DevChunk& Q, const DevChunk& R, const DevState& S, const DpLaunch& L,
                     const DpBuckets& B, const WorkQ& wq, int pgrid, hipStream_t st);
// score-only DP fills of nslots superpositions per pair (scores[k*np + p])
hipError_t launch_dp_score(const DevChunk& Q, const DevChunk& R, const DevState& S, int gap0, float gapopen,
                           const float* tfms, const int* slotflags, int nslots, float* scores, hipStream_t st);
// prec selects FP64 covariance and solve for the final-stage modes (FIN1,
// FIN2, PROD1, PROD2); DPREFINE is a search and stays FP32
hipError_t launch_refine_dp(int prec, int mode, const DevChunk& Q, const DevChunk& R,
                            const DevState& S, const Geom& G, const RefineLaunch& L, const RefSplit& Sp,
                            const WorkQ& wq, hipStream_t st);
// bytes of one part record (partbuf entries)
size_t part_record_bytes();
hipError_t launch_prod_aln(const DevChunk& Q, const DevChunk& R, const DevState& S, char* alns,
                           int nodel, const WorkQ& wq, int pgrid, hipStream_t st);
// work lists of live pairs (batched form): lista for the one-wave DP, listb for
// one-workgroup refinement, listc (optional) every live pair for the output
// pass; cnt holds 3 ints per 1024 pairs, totals 3 ints
hipError_t launch_live_lists(const DevState& S, const unsigned char* bigmask, int* cnt, int* totals, int* lista,
                             int* listb, int* listc, hipStream_t st);
// the pairs with alignment rows (tot: their number and packed bytes), and
// their rows packed
hipError_t launch_list_rows(const DevState& S, unsigned long long* tot, RowRec* recs, hipStream_t st);
hipError_t launch_pack_rows(const DevChunk& Q, const DevChunk& R, const DevState& S, const char* alns,
                            const RowRec* recs, size_t n, char* packed, hipStream_t st);
hipError_t launch_fill_i32(int* d, int v, size_t n, hipStream_t st);
// mixed precision: RMSD of every output pair's final alignment from FP64 sums
// and the quaternion matrix's largest eigenvalue (after the PROD1 refinement)
hipError_t launch_rmsd_fp64(const DevChunk& Q, const DevChunk& R, const DevState& S, hipStream_t st);
hipError_t launch_setlow(const DevChunk& Q, const DevChunk& R, const DevState& S, float thr,
                         hipStream_t st);
hipError_t launch_revert(const DevState& S, hipStream_t st);

}  // namespace gta
