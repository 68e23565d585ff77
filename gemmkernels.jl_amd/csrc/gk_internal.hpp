// Shared between the translation units of the host layer (not part of the C ABI).
#pragma once
#include <hip/hip_runtime.h>

#include "gemmkernels_hip.h"
#include "kernels/common.hpp"
#include "kernels/registry.hpp"

namespace gk_internal {

// Records the thread-local error message and returns `code`.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

struct Launch {
  gk::InstanceKey key;
  gk::InstanceInfo info;
  gk::GemmArgs args;
  int gx, gy;
  bool ragged;      // an aligned kernel runs bounds-checked layouts and has to take the last K tile out of its pipeline
};

int prepare_launch(const gk_config* conf, const void* a, const void* b, const void* c, void* d, const gk_transforms* transforms,
                   const gk_epilogue* epilogue, int32_t kernel, const gk::InstanceInfo* custom, Launch* out);

// The K-split launch on a workspace of `workspace_bytes` bytes at `workspace` ([arrival counters | partial tiles]);
// `whose` names the workspace in the message that refuses a launch it cannot hold.
int launch_split_k(const gk_config* conf, const void* a, const void* b, const void* c, void* d, const gk_transforms* transforms,
                   const gk_epilogue* epilogue, void* workspace, size_t workspace_bytes, const char* whose, void* stream);

}  // namespace gk_internal

// tail_chunk of every chunk of a tile on the host, with the code that the kernels inline, for tests of its arithmetic: `rows` x `cols` / 8 chunks, row by row
// (a K-major tile: rows of M or N, k along them; else rows of k).
extern "C" void gk_internal_tail_chunks(int32_t k_major, int32_t rows, int32_t cols, int32_t ld, int32_t rows_valid, int32_t tail_k, int32_t* from,
                                        int32_t* shift, int32_t* keep);
