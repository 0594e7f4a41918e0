// pair.h -- sweep kernel for vertices of degree <= 4 and bond dimensions <= 8 (complex: <= 5 on
// two bonds of a pair), FP64 or complex FP64, in the unpadded site layout of the generic kernel
// (kernel: pair.hip).
#pragma once

#include <string>
#include <vector>

#include "common.h"

#define PAIR_MAXD 8        // largest bond dimension
#define PAIR_SIDE 64       // largest pair dimension (two bonds of PAIR_MAXD)
#define PAIR_RUN_SWEEPS 256  // sweeps of one pair_run launch
#define PAIR_RUN_BAILED 2  // bit of the network's done flag: pair_run gave up

enum { PAIR_F64 = 0, PAIR_C128 = 1 };

// One vertex as the kernel reads it.  Its ports are split into two pairs of consecutive
// tensor axes, positions (0, 1) and (2, 3): degree 4 (p0 p1)(p2 p3), degree 3 (p0 p1)(p2),
// degree 2 (p0)(p1), degree 1 (p0)().  An absent position has dimension 1 and slot -1.
struct PairRec {
    long long site;     // element offset of the site tensor
    long long in[4];    // element offset of the incoming message per position
    long long out[4];   // element offset of the outgoing message
    int slot[4];        // outgoing message slot
    int dim[4];
    int d, net;
    int n[2];           // pair dimensions dim[0] dim[1], dim[2] dim[3]
    int vertex, pad;
};

struct PairPlan {
    int dtype = PAIR_F64;
    std::vector<PairRec> recs;       // one per vertex of positive degree
    std::vector<int> rec_of;         // vertex -> record, -1 when the vertex does not qualify
    std::vector<int> rest;           // message slots of the other vertices
    PairRec *d_recs = nullptr;
    int *d_lead = nullptr;           // per network: its first record
    bool covers = false;             // it takes every message of every network
    bool all = false;                // and every vertex (no isolated ones)
    int nt = 0;                      // 16-wide tiles of the largest pair dimension
    int chunk = 0, split = 0;        // slices staged in LDS at once; waves sharing a tile's slices
    int waves = 0;
    int slice_elems = 0, env_elems = 0;  // LDS elements per plane
    size_t lds_bytes = 0;

    // many sweeps a launch (pair_run): allocated on first use for the plan's life, at most
    // 8 versions of the messages of a network that fits the device at once
    int run_state = 0;               // 0: not looked at, 1: ready, -1: not for this network
    int run_pause = 0, run_next = 0; // runs to leave out, twice the next pause
    long long run_nm = 0;            // doubles of one version
    int run_nports = 0;
    void *d_run = nullptr;                 // what the pointers below point into
    int *d_steps[2] = {nullptr, nullptr};  // Jacobi, sequential
    void *d_ring = nullptr, *d_ctrl = nullptr;
    double *d_ring_res = nullptr;
};

void pair_release(PairPlan *p);
// 0 on success, 4 when no vertex qualifies, other values on a device error
int pair_plan_build(PairPlan *p, int dtype, int plain, int nv, int nnet, const int *port_off,
                    const int *port_edge, const int *edge_dim, const int *phys_dim,
                    const int *port_rev, const int *vnet, const long long *site_off,
                    const long long *msg_off);
// 16x16x4 products per physical slice of a vertex, on average: the kernel's time grows with it
double pair_mfma_per_slice(const PairPlan *p);
// One launch over records [0, n) when `items` is null (every message of every record), else
// over n work items of `items` (record * 4 + position: one message each).  src == dst is
// allowed for messages that no work item of the launch reads.
int pair_sweep(const PairPlan *p, hipStream_t st, const void *sites, const void *src, void *dst,
               const NetCtl &ctl, double *res_fid, double *res_abs, const SweepFold &fold,
               const int *items = nullptr, int n = 0);
// Vertex scalars of every record at the messages `msgs`: zv[vertex] (complex: interleaved).
int pair_scalars(const PairPlan *p, hipStream_t st, const void *sites, const void *msgs,
                 double *zv);

// Many sweeps of one network in a launch, its vertices resident together: whether the plan
// takes it (and its buffers are there).
bool pair_run_ready(PairPlan *p, int nnet, long long nmsg, int nports);
// After a run that gave up, the next 1, 2, 4, .. runs are left out (the count starts again after
// one that did not): whether this one is, and how one that was not has ended.
bool pair_run_paused(PairPlan *p);
void pair_run_ended(PairPlan *p, bool gave_up);
// The schedule of sequential runs, [record][4]: positions | versions << 4 (see pair.hip).
int pair_run_steps(PairPlan *p, hipStream_t st, const std::vector<int> &steps);
// `sweeps` sweeps from src to dst (src is left as it is), `first` already done; the network's
// state and residuals as after a folded run.  done & PAIR_RUN_BAILED: nothing is valid, run
// again launch by launch (a wait in the kernel took longer than wait_us).  One launch at a time
// per device: two that wait for each other's room would both give up.
int pair_run(const PairPlan *p, hipStream_t st, bool sequential, const void *sites,
             const void *src, void *dst, int *done, int *iter, int *at, double *delta,
             double *res_fid, double *res_abs, const RunParams &rp, int first, int sweeps,
             int wait_us);
