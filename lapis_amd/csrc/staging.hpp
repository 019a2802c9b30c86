// Operands of one call that come from and go back to ordinary host memory; see staging.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <vector>

#include "plan.hpp"

namespace lapis {

struct StagingArena;

class HostOperands {
 public:
  HostOperands() = default;
  ~HostOperands();  // waits for what an early exit left queued
  HostOperands(const HostOperands &) = delete;
  HostOperands &operator=(const HostOperands &) = delete;

  // Announce the operands; each gets an index.  A null `host` is device memory only.
  int add(const void *host, size_t bytes);
  // An operand that kernels read and write once per element: up to kDirect bytes of it stay in pinned memory.
  int add_direct(const void *host, size_t bytes);
  // The positions and the coordinates of a CSR structure: the pass that copies them also checks and counts them.
  int add_positions(const int32_t *host, int64_t nrows, int64_t nnz);
  int add_coordinates(const int32_t *host, int64_t nnz, int64_t ncols);

  // The copies and what follows are queued on this stream instead of one of the arena's own.
  void use_stream(hipStream_t st) {
    primary_ = st;
    own_stream_ = false;
  }

  int create_plan(int positions, int coordinates, int value_bytes, lapis_hip_csr_plan **plan);  // after upload()

  int upload();  // takes memory for all of them and queues their copies on stream()
  template <typename T>
  T *at(int index) const {
    return static_cast<T *>(device(index));
  }
  hipStream_t stream() const { return primary_; }
  lapis_hip_stream_t abi_stream() const { return reinterpret_cast<lapis_hip_stream_t>(stream()); }

  // Brings an operand's device memory to `host`, after what is queued on stream(); returns when it is there.
  int download(int index, void *host);
  int download(const void *from, size_t bytes, void *host);  // the same for any device memory
  int synchronize();

  struct Block {  // what one thread copies at a time
    char *staged;
    char *host;
    size_t bytes, at;  // at: from the start of the operand
    int operand;
    size_t end;  // where it ends in the device memory of the call
  };
  void copy_block(const Block &b, bool to_host);

 private:
  enum Kind { kPlain, kCoordinates, kPositions, kDeviceOnly, kDirectly };  // in the order in which they lie in memory
  struct Operand {
    const char *host;
    size_t bytes, at;
    Kind kind;
  };
  void *device(int index) const;

  std::vector<Operand> operands_;
  size_t bytes_ = 0;
  StagingArena *arena_ = nullptr;
  hipStream_t primary_ = nullptr;
  bool own_stream_ = true;
  bool idle_ = true;  // nothing is queued on the stream
  CsrCounts counts_{};  // of the CSR structure, after upload()
  int64_t nrows_ = 0, nnz_ = 0, ncols_ = 0;
};

void release_staging();  // memory and threads kept between calls

}  // namespace lapis
