// hg_resident.hpp -- resident runs: many steps (or right-hand sides, or
// reverse steps) of a small mesh in one launch (hg_resident.hip), as the
// rest of the library calls them.
#pragma once
#include <hip/hip_runtime.h>

#include "hg_ctx.hpp"

namespace hg {

constexpr int kResT = 128;           // cells per tile
constexpr int64_t kResSteps = 4096;  // steps per launch
constexpr int64_t kResTrials = 1024; // Tsit5 trial steps per launch
constexpr int kResRed = 256;         // tiles a run with a reduction over them may have

// Work items a tile may hold: one per work-item of its work-group.
constexpr int res_items(int MD) { return MD == 3 ? 256 : 320; }

// Where Manning's n (or the friction magnitude) comes from.
enum { RES_N_FIELD = 0, RES_N_LAW = 1, RES_N_NET = 2 };

struct ResArgs {
  unsigned long long* ring;  // [4][3][N] ([4][6][N] with tangents)
  int32_t* ctl;              // [0]: a wait ran out
  int64_t ns;                // steps
  const int32_t* nbr;        // ELL, for the published cells
  // optional record of the run (the adjoint's forward sweep): states 0 .. ns
  // ([ns + 1][3][N]; state 0 is there already), clamps [ns][N], conveyances
  // and, with a law or network, its n of each step [ns][N]
  double* rec;
  uint8_t* rec_clamp;
  double* rec_totalA;
  double* rec_n;
  int32_t n_inlet;
  // variable-n law, or the UDE network (its output is the friction magnitude
  // for HG_LUX_FLOW_RESISTANCE), with their per-cell ks
  NLaw law;
  LuxNet net;
  const double* ks;
  const double* net_w;
  // forward mode: tangents of the state in and out, of the parameter fields
  // and of the network's weights (NULL: zero)
  const double *dxi, *dqx, *dqy;
  double *dxo, *dqxo, *dqyo;
  const double *dn, *dzb, *dS0x, *dS0y, *dg_zb, *dinletQ, *net_dw;
};

// An adaptive Tsit5 run: the solver's state between launches, and its output.
struct Tsit5State {
  double t, dt;
  int64_t frame, accepted, rejected, nrhs;  // frame: the one being integrated towards (1 .. n_save)
  int32_t code;  // HG_OK, or why it stopped: HG_ERR_NONFINITE (error estimate), HG_ERR_STATE (1: underflow, 2: too many steps in sub)
  int32_t sub;
  int32_t done;
};
struct Tsit5Args {
  double t0, t1, abstol, reltol;
  int64_t n_save, trials, max_steps;
  const Tsit5State* in;       // NULL: the start (t0, dt0)
  double dt0;
  Tsit5State* out;
  double* y;                  // [3][N] solution between launches (in and out)
  double* k0;                 // [3][N] its derivative
  unsigned long long* red;    // [4][kResRed] the tiles' error sums
  double* frames;             // [n_save + 1][3][N] in caller order; frame 0 is written by the first launch
  const int32_t* perm;
};

// Reverse mode of a recorded run.
struct AdjRunArgs {
  unsigned long long* ring;   // [4][3][N] cotangents
  unsigned long long* vring;  // [4][G] inlet ghost velocity cotangents
  int32_t* ctl;
  int32_t* flag;              // the host's error flags
  int64_t ns, G;
  const double* rec;          // [ns][3][N] states
  const uint8_t* rec_clamp;   // [ns][N]
  const double* rec_totalA;   // [ns][n_inlet]
  int32_t n_inlet;
  const int32_t* tile_in_off;
  const int32_t* tile_in_list;
  const int32_t* in_off;
  const InletFaceRec* in_rec;
  const double* Qbar;
  double *o_nbar, *o_zbbar, *o_S0bar, *o_Qbar;  // o_Qbar: of the inlets that have faces
  // with a law or network: what the forward run recorded of it ([ns][N]), the
  // closure (as in ResArgs), and the tiles' weight cotangents ([P][ntiles])
  const double* rec_n;
  NLaw law;
  LuxNet net;
  const double* ks;
  const double* net_w;
  double* o_wpart;
};

// The kernel variants.  split: the cells' work-items take no items (few tiles).
struct ResKind {
  int md;      // 3 or 4
  bool split;
  int nmode;   // RES_N_*
  bool dual;   // with tangents
};

// Tiles of such a run that the device surely holds at once (0: there is no
// such variant).
int res_capacity(const ResKind& k, int ncu);
int adj_run_capacity(int md, int nmode, int net_P, int ncu);
// Weights and hidden layers a resident reverse run can hold (2 LDS values per weight and cell).
constexpr int kAdjRunMaxP = 56, kAdjRunMaxHidden = 2;
// Tiles of a mesh on which such a network's weight cotangents are summed cell by cell, resident or not.
constexpr int kAdjRunNetTiles = 256;
int tsit5_capacity(int md, int nmode, int ncu);

hipError_t res_init(hipStream_t stream, int64_t n, unsigned long long* ring, int32_t* ctl);
hipError_t launch_run(hipStream_t stream, const ResKind& k, int ntiles, const TileArgs& a, const ResArgs& R);
hipError_t launch_adj_run(hipStream_t stream, int md, int nmode, int ntiles, const AdjArgs& a, const AdjRunArgs& R);
hipError_t launch_tsit5(hipStream_t stream, int md, int nmode, int ntiles, const TileArgs& a, const ResArgs& R,
                        const Tsit5Args& P);

}  // namespace hg
