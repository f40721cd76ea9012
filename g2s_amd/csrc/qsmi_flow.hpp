// Data-flow path loop (qsmi_flow.hip): what the host layer hands over.
#pragma once
#include "qsmi_internal.hpp"

namespace qsmi {

constexpr int kFlowMaxTerms = 512;  // n x variables
constexpr int kFlowMaxCat = 16;     // classes of all variables
constexpr int kFlowQuant = 128;     // quantiles of a continuous variable

struct FlowPlan {
  bool count = false;  // categorical variables, one weight: bit-sliced counts
  bool mixed = false;  // direct form with a categorical variable
  bool unitW = false;  // every kernel weight is 1
  long long nPath = 0;
  int nClasses = 0;
  int e0[8] = {}, nCat[8] = {}, cat0[8] = {};  // per variable: first expanded index, classes, first class
  std::vector<float> quant;                    // [variable][kFlowQuant] quantiles of the continuous variables
  float rare[kFlowMaxCat] = {};                // per class: 1 - its share of the TI
  int inFlight = 1 << 20;  // path nodes simulated at the same time, at most
  int segment = 65536;     // path nodes per launch
  bool alone = false;      // the whole path, whatever the waves would take
  // what the wave loop takes, microseconds: a wave, a node, its spectra and
  // buffers (waveNodeUs 0: the path is never handed over to it)
  double waveUs = 0.0, waveNodeUs = 0.0, waveSetupUs = 0.0;
};

// Simulates the path (R's neighbour lists, grid and tables on the device).
// stats: exact-selection nodes, rescored positions, 0, list flushes.
// done: nodes of R's order that are simulated, in the grid and the index image;
// the rest, if any, is faster by waves.
// gaveUp: a wait hit its bound; the grid is not usable then.
int run_flow(qsmi_ti* t, const ResidentLoop& R, const FlowPlan& F, double* kernelMs, long long* stats, size_t* done,
             bool* gaveUp);

}  // namespace qsmi
