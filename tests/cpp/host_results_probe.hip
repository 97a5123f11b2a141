// The host side of results on their way (nd_host_results.hpp), on a machine without a GPU: what is asked for is the first argument.
//   exit     the process ends while one of the threads is at work: prints "ended 1" if that work was waited for
//   fork     a child forked while one of the threads is at work ends at once: prints "child ended 1"
//   cpus     CPUs that the control groups under a folder give a process whose groups a file lists (two more arguments)
//   threads  threads that took part in something
//   pool     bytes that wait for their next use after arrays were given back, after a trim, and at the end
#include "../../nextdoor_amd/csrc/nd_host_results.hpp"

#include <stdio.h>
#include <sys/wait.h>

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

static int fork_while_at_work() {
  exit_while_at_work();
  const pid_t child = fork();
  if (child < 0) return 1;
  if (child == 0) exit(0);
  const auto t0 = std::chrono::steady_clock::now();
  int status = -1;
  if (waitpid(child, &status, 0) != child) return 1;
  const bool soon = std::chrono::steady_clock::now() - t0 < std::chrono::seconds(5);
  printf("child ended %d\n", status == 0 && soon);
  return 0;
}

static int threads_that_take_part() {
  std::mutex mutex;
  std::vector<std::thread::id> seen;
  nd::HostWorkers::get().run(nd::HostWorkers::kMost, [&] {
    {
      std::lock_guard<std::mutex> lock(mutex);
      seen.push_back(std::this_thread::get_id());
    }
    std::this_thread::sleep_for(std::chrono::milliseconds(300));
  });
  printf("%zu\n", seen.size());
  return 0;
}

static int arrays_that_wait() {
  auto pool = std::make_shared<nd::HostPool>();
  std::vector<nd::HostBlock> held;
  for (int i = 0; i < 5; ++i) held.push_back(pool->take(16u << 20));
  for (const nd::HostBlock& b : held) pool->give(b);
  printf("%zu\n", pool->waiting_bytes());
  for (size_t kinds = 1; kinds <= 4; ++kinds) {  // of a walk without states; of edge lists with all there is
    pool->keep(kinds);
    for (nd::HostBlock& b : held) b = pool->take(16u << 20);
    for (const nd::HostBlock& b : held) pool->give(b);
    printf("%zu\n", pool->waiting_bytes());
  }
  pool->trim();
  printf("%zu\n", pool->waiting_bytes());
  nd::HostBlock last = pool->take(1000);
  pool->give(last);
  printf("%zu\n", pool->waiting_bytes());
  last = pool->take(1000);
  pool->close();
  pool->give(last);
  printf("%zu\n", pool->waiting_bytes());
  return 0;
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "exit") return exit_while_at_work();
  if (what == "fork") return fork_while_at_work();
  if (what == "cpus" && argc > 3) return printf("%g\n", nd::cpus_of_groups(argv[2], argv[3])) < 0;
  if (what == "pool") return arrays_that_wait();
  if (what == "threads") return threads_that_take_part();
  return 2;
}
