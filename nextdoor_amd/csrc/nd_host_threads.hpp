// How many threads of the host this process may keep busy.
#pragma once

#include <math.h>
#include <stdlib.h>

#include <algorithm>
#include <fstream>
#include <sstream>
#include <string>
#include <thread>

namespace nd {

// CPUs' worth of time the control group with these files is given; infinity: no limit, or no such group.
inline double cpus_of_group(const std::string& dir) {
  std::string quota;
  double period = 0;
  if (std::ifstream(dir + "/cpu.max") >> quota >> period) {  // "max 100000" or "1600000 100000"
    const double q = atof(quota.c_str());
    return q > 0 && period > 0 ? q / period : INFINITY;
  }
  double q = 0;
  if (std::ifstream(dir + "/cpu.cfs_quota_us") >> q && std::ifstream(dir + "/cpu.cfs_period_us") >> period && q > 0 && period > 0)
    return q / period;
  return INFINITY;
}

// The same for the process whose groups are listed in `groups_file`, under the control groups mounted at `root`: the
// least of its own group's and of all that group is part of.
inline double cpus_of_groups(const std::string& root, const std::string& groups_file) {
  double least = std::min(cpus_of_group(root), cpus_of_group(root + "/cpu"));
  std::ifstream groups(groups_file);
  for (std::string line; std::getline(groups, line);) {  // hierarchy:controllers:path
    const size_t a = line.find(':'), b = a == std::string::npos ? a : line.find(':', a + 1);
    if (b == std::string::npos) continue;
    const std::string controllers = "," + line.substr(a + 1, b - a - 1) + ",";
    if (controllers != ",," && controllers.find(",cpu,") == std::string::npos) continue;
    const std::string base = controllers == ",," ? root : root + "/cpu";
    for (std::string path = line.substr(b + 1); path.size() > 1; path.resize(path.rfind('/')))
      least = std::min(least, cpus_of_group(base + path));
  }
  return least;
}

// CPUs of this process: those the scheduler may put it on (which hardware_concurrency() counts), and no more than its
// control group gives it time for (which it does not know of: a container with 4 CPUs' time on 256 runs threads 250 of which wait).
inline unsigned host_cpus() {
  static const unsigned cpus = [] {
    const unsigned seen = std::thread::hardware_concurrency(), here = seen ? seen : 4;  // 0: it cannot tell
    const double given = std::ceil(cpus_of_groups("/sys/fs/cgroup", "/proc/self/cgroup"));
    return given < here ? std::max(1u, (unsigned)given) : here;
  }();
  return cpus;
}

// ND_HOST_THREADS, or 0
inline unsigned host_threads_wanted() {
  const char* env = getenv("ND_HOST_THREADS");
  const int v = env ? atoi(env) : 0;
  return v > 0 ? (unsigned)v : 0u;
}

// Threads for work that any number can take part in: as many as are asked for, or one a CPU but no more than `most`.
inline unsigned host_threads(unsigned most) {
  const unsigned wanted = host_threads_wanted();
  return wanted ? wanted : std::min(host_cpus(), most);
}

}  // namespace nd
