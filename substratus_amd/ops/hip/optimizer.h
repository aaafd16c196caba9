// Arguments of the optimizer's kernels: tensors by value, so that a launch
// needs no table copied to the device before it.
#pragma once

// One launch's tensors; 40 of them stay below the 4 KiB of a launch's
// arguments.
constexpr int OPT_MOST = 40;

struct OptTensor {
  void* p;          // parameter (unused by the norm)
  const void* g;    // its gradient
  float *m, *v;     // moments (unused by the norm)
  long n;           // elements
  int block;        // first workgroup
};

struct OptTensors {
  OptTensor t[OPT_MOST];
  int count;
};
