// Host work beside the calling thread.
#pragma once
#include <future>
#include <system_error>
#include <utility>
#include <vector>

namespace fgpu {

// Jobs on threads of their own, each waited for on every way out.  What a job
// refers to is declared before the HostJobs object, so that it outlives the
// job where an error leaves the scope.  A job that no thread is to be had for
// is done at once by the caller.
class HostJobs {
 public:
  template <class F>
  void start(F job) {
    std::future<void> f;
    try {
      f = std::async(std::launch::async, job);
    } catch (const std::system_error&) {
      job();
      return;
    }
    jobs_.push_back(std::move(f));
  }
  void wait() {
    for (auto& f : jobs_) f.get();
    jobs_.clear();
  }

 private:
  std::vector<std::future<void>> jobs_;
};

}  // namespace fgpu
