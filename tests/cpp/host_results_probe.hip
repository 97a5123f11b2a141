// The host side of results on their way (nd_host_results.hpp), on a machine without a GPU: what is asked for is the first argument.
//   exit     the process ends while one of the threads is at work: prints "ended 1" if that work was waited for
#include "../../nextdoor_amd/csrc/nd_host_results.hpp"

#include <stdio.h>

static std::atomic<int> begun(0), ended(0);
static nd::HostWorkers::Job job;

static int exit_while_at_work() {
  // registered before the threads are: runs after what they registered, as the HIP runtime's own does
  atexit([] { printf("ended %d\n", ended.load()); });
  job.body = [] {
    begun++;
    std::this_thread::sleep_for(std::chrono::milliseconds(300));
    ended++;
  };
  nd::HostWorkers::get().start(job, 1);
  while (begun.load() == 0) std::this_thread::yield();
  return 0;
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "exit") return exit_while_at_work();
  return 2;
}
