/* A stand-in for the part of the HIP runtime that a kernel launch uses, loaded ahead of it: launches do
 * nothing and are counted, and the launch whose number is llmopt_stub_fail fails as the runtime's do --
 * its error stays until hipGetLastError is asked, which clears it. */
#include <stddef.h>

typedef struct { unsigned x, y, z; } dim3_t;

int llmopt_stub_launches = 0;
int llmopt_stub_fail = 0;
static int last_error = 0;
static dim3_t grid_, block_;
static size_t shared_;
static void* stream_;

int __hipPushCallConfiguration(dim3_t grid, dim3_t block, size_t shared, void* stream) {
  grid_ = grid, block_ = block, shared_ = shared, stream_ = stream;
  return 0;
}

int __hipPopCallConfiguration(dim3_t* grid, dim3_t* block, size_t* shared, void** stream) {
  *grid = grid_, *block = block_, *shared = shared_, *stream = stream_;
  return 0;
}

int hipLaunchKernel(const void* f, dim3_t grid, dim3_t block, void** args, size_t shared, void* stream) {
  (void)f, (void)grid, (void)block, (void)args, (void)shared, (void)stream;
  if (++llmopt_stub_launches != llmopt_stub_fail) return 0;
  return last_error = 1; /* hipErrorInvalidValue */
}

int hipGetLastError(void) {
  const int e = last_error;
  last_error = 0;
  return e;
}

int hipFuncSetAttribute(const void* f, int attribute, int value) {
  (void)f, (void)attribute, (void)value;
  return 0;
}
