// What a launch costs on the GPU at hand, whatever the kernel does: the floor under the latency
// of the decode-sized steps, whose two kernels run for 4-6 us each.
//
// Empty kernels of 256 workgroups of 1024 threads are launched as the library launches its own
// (launch_kernel), with as many bytes of arguments as its kernels have: 104 beside a table in
// device memory, 176 in the routing, 1240 with a rank table of up to eight ranks, 9304 with one of
// 64.  They are timed three ways, back to back on one stream: eager launches, replays of a
// captured graph holding one such kernel, and replays of a graph holding two.  Two figures per
// line: microseconds per launch (or replay) on the GPU's side, from HIP events around the whole
// batch, and microseconds of host time per call.  Then the host time of an eager launch again,
// by launch_kernel and by <<<>>> in turn, the median of nine batches of each.
//
//   bench_launch [batch]       (default 2000 launches per figure)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>

#include "a2a_common.h"

#define HIP_OK(expr)                                                                       \
  do {                                                                                     \
    hipError_t e_ = (expr);                                                                \
    if (e_ != hipSuccess) {                                                                \
      fprintf(stderr, "%s failed: %s\n", #expr, hipGetErrorString(e_));                    \
      exit(1);                                                                             \
    }                                                                                      \
  } while (0)

template <int BYTES> struct Arguments {  // (beside the pointer)
  unsigned long long v[BYTES / 8 - 1];
};

template <class Args>
__global__ void empty_kernel(Args a, unsigned long long *sink) {
  // (never true: keeps the arguments alive without touching memory)
  if (a.v[0] == 0x5555aaaa5555aaaaull && threadIdx.x == 4096) sink[0] = a.v[1];
}

struct Figure {
  double gpu_us, host_us;
};

template <class Launch>
Figure time_batch(hipStream_t stream, int batch, Launch launch) {
  hipEvent_t start, stop;
  HIP_OK(hipEventCreate(&start));
  HIP_OK(hipEventCreate(&stop));
  for (int i = 0; i < 50; ++i) launch();
  HIP_OK(hipStreamSynchronize(stream));
  HIP_OK(hipEventRecord(start, stream));
  const auto t0 = std::chrono::steady_clock::now();
  for (int i = 0; i < batch; ++i) launch();
  const auto t1 = std::chrono::steady_clock::now();
  HIP_OK(hipEventRecord(stop, stream));
  HIP_OK(hipStreamSynchronize(stream));
  float ms = 0.f;
  HIP_OK(hipEventElapsedTime(&ms, start, stop));
  HIP_OK(hipEventDestroy(start));
  HIP_OK(hipEventDestroy(stop));
  return Figure{ms * 1e3 / batch, std::chrono::duration<double, std::micro>(t1 - t0).count() / batch};
}

template <class Args>
void run(const char *what, dim3 grid, dim3 block, hipStream_t stream, int batch, unsigned long long *sink) {
  Args args{};
  auto eager = [&] {
    HIP_OK((hipError_t)pplx_amd::launch_kernel(empty_kernel<Args>, grid, block, 0, stream, args, sink));
  };
  const Figure e = time_batch(stream, batch, eager);
  Figure g[2];
  for (int nodes = 1; nodes <= 2; ++nodes) {
    hipGraph_t graph;
    hipGraphExec_t exec;
    HIP_OK(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
    for (int i = 0; i < nodes; ++i) eager();
    HIP_OK(hipStreamEndCapture(stream, &graph));
    HIP_OK(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    g[nodes - 1] = time_batch(stream, batch, [&] { HIP_OK(hipGraphLaunch(exec, stream)); });
    HIP_OK(hipGraphExecDestroy(exec));
    HIP_OK(hipGraphDestroy(graph));
  }
  // two eager launches per "step", for comparison with the two-node graph
  const Figure e2 = time_batch(stream, batch, [&] { eager(); eager(); });
  printf("%-44s %8.2f %8.2f   %8.2f %8.2f   %8.2f %8.2f   %8.2f %8.2f\n", what, e.gpu_us, e.host_us, e2.gpu_us,
         e2.host_us, g[0].gpu_us, g[0].host_us, g[1].gpu_us, g[1].host_us);
}

// Host time of an eager launch, either way.
template <class Args>
void compare(hipStream_t stream, int batch, unsigned long long *sink) {
  constexpr int kBatches = 9;
  const dim3 grid(256), block(1024);
  Args args{};
  double ours[kBatches], theirs[kBatches];
  for (int i = 0; i < kBatches; ++i) {
    ours[i] = time_batch(stream, batch, [&] {
                HIP_OK((hipError_t)pplx_amd::launch_kernel(empty_kernel<Args>, grid, block, 0, stream, args, sink));
              }).host_us;
    theirs[i] = time_batch(stream, batch, [&] {
                  empty_kernel<Args><<<grid, block, 0, stream>>>(args, sink);
                }).host_us;
  }
  std::sort(ours, ours + kBatches);
  std::sort(theirs, theirs + kBatches);
  printf("%6zu bytes   launch_kernel %6.2f   <<<>>> %6.2f\n", sizeof(Args) + sizeof(sink), ours[kBatches / 2],
         theirs[kBatches / 2]);
}

int main(int argc, char **argv) {
  const int batch = argc > 1 ? atoi(argv[1]) : 2000;
  int n_dev = 0;
  if (hipGetDeviceCount(&n_dev) != hipSuccess || n_dev == 0) {
    fprintf(stderr, "bench_launch: no GPU visible\n");
    return 2;
  }
  HIP_OK(hipSetDevice(0));
  hipStream_t stream;
  HIP_OK(hipStreamCreate(&stream));
  unsigned long long *sink;
  HIP_OK(hipMalloc(&sink, 64));
  printf("empty kernels, %d launches (or replays) per figure, back to back on one stream; us per call: GPU side / host side\n",
         batch);
  printf("%-44s %17s   %17s   %17s   %17s\n", "kernel", "1 eager launch", "2 eager launches", "graph of 1 node",
         "graph of 2 nodes");
  run<Arguments<104>>("104 bytes of arguments", dim3(256), dim3(1024), stream, batch, sink);
  run<Arguments<176>>("176 bytes of arguments", dim3(256), dim3(1024), stream, batch, sink);
  run<Arguments<1240>>("1240 bytes of arguments", dim3(256), dim3(1024), stream, batch, sink);
  run<Arguments<9304>>("9304 bytes of arguments", dim3(256), dim3(1024), stream, batch, sink);
  printf("\nhost us per eager launch\n");
  compare<Arguments<104>>(stream, batch, sink);
  compare<Arguments<176>>(stream, batch, sink);
  compare<Arguments<1240>>(stream, batch, sink);
  compare<Arguments<9304>>(stream, batch, sink);
  HIP_OK(hipFree(sink));
  HIP_OK(hipStreamDestroy(stream));
  return 0;
}
