// KNCustomizedOp: a kernel-level operator whose body is a thread-block graph
// (reference include/mirage/kernel/customized.h:28-45).
#pragma once

#include "mirage/kernel/operator.h"
#include "mirage/threadblock/graph.h"
#include <memory>

namespace mirage {
namespace kernel {

struct KeptLaunch;

class KNCustomizedOp : public KNOperator {
public:
  // Builds the thread-block graph from a plan: one input loader per tensor, the
  // plan's operators in order, then one accumulating output per tile that no
  // later operator consumes (reference src/kernel/customized.cc:65-186).
  // (by value: a caller that has no more use for them moves them in)
  KNCustomizedOp(std::vector<DTensor> inputs, mirage::threadblock::ExecutionPlan plan);
  // Rebuilds an existing thread-block graph over new inputs and recovers its plan.
  KNCustomizedOp(std::vector<DTensor> const &inputs, mirage::threadblock::Graph const &_graph);
  virtual ~KNCustomizedOp();
  bool profile(ProfileResult &profile) override;
  void run(void);  // one fp16 launch on the backend stream, no synchronisation
  void run_with(KNCustomizedOp &next);  // run(), next.run()
  bool fingerprint(void) override;
  operator json() const override;  // adds bgraph and plan (src/kernel/customized.cc:315-321)

  mirage::threadblock::ExecutionPlan plan;
  mirage::threadblock::Graph bgraph;

private:
  // the kernel launches of run() [0] and fingerprint() [1] per backend queue, kept from one call
  // to the next
  std::shared_ptr<KeptLaunch> kept[2][4];
  std::shared_ptr<KeptLaunch> kept_two[4];  // of run() and the next operator's together (execute_all)
  void launch(bool fingerprint);
  void add_output(mirage::threadblock::STensor const &stensor, int3 output_map);
};

}  // namespace kernel
}  // namespace mirage
