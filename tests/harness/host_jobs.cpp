// fgpu::HostJobs where threads run out: argv[1] starts succeed, the others
// fail as pthread_create does at a process limit.  Prints "jobs done, threads
// started"; a job that throws is reported by wait().
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <stdexcept>
#include <string>
#include <thread>
#include "../../fedem-solvers_amd/csrc/host_jobs.hpp"

static int allowed, started;

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*run)(void*), void* arg) {
  using Create = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static Create real = reinterpret_cast<Create>(dlsym(RTLD_NEXT, "pthread_create"));
  if (started >= allowed) return EAGAIN;
  started++;
  return real(t, a, run, arg);
}

int main(int argc, char** argv) {
  allowed = argc > 1 ? std::atoi(argv[1]) : 0;
  const bool fail = argc > 2;
  std::vector<int> out(5, 0);
  std::string err;
  try {
    fgpu::HostJobs jobs;
    for (int i = 0; i < 5; i++)
      jobs.start([&out, i, fail]() {
        std::this_thread::sleep_for(std::chrono::milliseconds(20));
        out[i] = 1;
        if (fail && i == 1) throw std::runtime_error("job 1");
      });
    jobs.wait();
  } catch (const std::exception& e) {
    err = e.what();  // every job that was started has ended
  }
  int done = 0;
  for (int v : out) done += v;
  std::printf("%d %d %s\n", done, started, err.c_str());
  return 0;
}
