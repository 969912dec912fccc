// jk_lanes.h -- the class launches of a J/K build over four streams.
//
// The 21 class kernels of a build are independent.  Where they do not fill the
// chip (a small molecule) their latencies would add up on one or two streams, and where they do, each kernel's last
// workgroups leave room for the next lane's: a process has four hardware queues,
// so four lanes.  Each class goes to the lane with the least time so far, longest
// class first, by an estimate of 50 us a kernel and 0.1 us a primitive step of
// its longest job's waves and of its share of 2048 resident waves.  A batch's
// builds run so, and the captured graph of one molecule's, which is made at the
// second build with one set of outputs: the first (water / 6-31G* 0.93 ms) is
// launched over two streams.  A server keeps to two as well (bscf.hip).
// Measured in the captured graph of a build, two streams -> four lanes: water /
// 6-31G* 0.84 -> 0.56 ms, (H2O)4 / cc-pVDZ 1.79 -> 1.34, (H2O)8 4.16 -> 3.78,
// (H2O)16 16.3 -> 15.9, C10H22 / def2-SVP 3.19 -> 2.75.
#pragma once
#include <hip/hip_runtime.h>

#include "engine.h"

namespace hfg {

struct JKLanes {
  static constexpr int N = 4;
  hipStream_t s[N] = {};  // s[0]: the caller's
  hipEvent_t ev[2 * (N - 1)] = {};
  explicit JKLanes(hipStream_t main);
  ~JKLanes();
  JKLanes(const JKLanes&) = delete;
  JKLanes& operator=(const JKLanes&) = delete;
};
// Cost of each class's jobs (plan.job_cost units): the longest and all together.
struct JKClassCost {
  double longest[HFG_NCLASS] = {}, sum[HFG_NCLASS] = {};
  void add(const JKPlan& plan);
  void add(const JKClassCost& c);
};
void assign_lanes(const JKClassCost& cost, int (&lane)[HFG_NCLASS]);

// The class launches over streams s[0 .. count): lane[c] and cap[c] are class c's
// stream and workgroup cap.  The other lanes start after s[0]'s earlier work and
// are joined to it at the end (events ev[2 k - 2], ev[2 k - 1] for lane k).
void launch_jk_lanes(const JKLaunch& L, const MolTab* d_tabs, const JKDirectory& dir, const int* d_dir,
                     const hipStream_t* s, const hipEvent_t* ev, int count, const int* lane, const int* cap);

}  // namespace hfg
