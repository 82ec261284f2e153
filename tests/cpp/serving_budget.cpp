// Device memory of the serving loop, counted on the host: this program
// defines the HIP runtime calls that libdgops.so makes (host memory for the
// device's, nothing for launches, streams and events), so the library's own
// admission and buffer handling run without a GPU.
//
//   serving_budget
//
// prints, in bytes: the budget and the peak of the device memory while
// requests of another size follow finished ones whose buffers are idle, the
// number of new device blocks that the same request takes a second time, and
// the memory in use after the server is gone.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

#include <hip/hip_runtime.h>

#include "dgops.h"

static std::map<void *, size_t> blocks;
static size_t                   live = 0, peak = 0;
static int                      n_malloc = 0;

extern "C" {

hipError_t
hipMalloc(void **p, size_t bytes)
{
  *p = std::calloc(1, bytes);
  blocks[*p] = bytes;
  live += bytes;
  if (live > peak)
    peak = live;
  ++n_malloc;
  return hipSuccess;
}
hipError_t
hipFree(void *p)
{
  if (!p)
    return hipSuccess;
  live -= blocks.at(p);
  blocks.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t
hipHostMalloc(void **p, size_t bytes, unsigned)
{
  *p = std::malloc(bytes);
  return hipSuccess;
}
hipError_t
hipHostFree(void *p)
{
  std::free(p);
  return hipSuccess;
}
hipError_t
hipMemcpy(void *d, const void *s, size_t bytes, hipMemcpyKind)
{
  std::memcpy(d, s, bytes);
  return hipSuccess;
}
hipError_t
hipMemcpyAsync(void *d, const void *s, size_t bytes, hipMemcpyKind,
               hipStream_t)
{
  std::memcpy(d, s, bytes);
  return hipSuccess;
}
hipError_t
hipGetDevice(int *d)
{
  *d = 0;
  return hipSuccess;
}
hipError_t
hipGetLastError()
{
  return hipSuccess;
}
hipError_t
hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t)
{
  return hipSuccess;
}
hipError_t
hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
  *s = nullptr;
  return hipSuccess;
}
hipError_t
hipStreamDestroy(hipStream_t)
{
  return hipSuccess;
}
hipError_t
hipStreamSynchronize(hipStream_t)
{
  return hipSuccess;
}
hipError_t
hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned)
{
  return hipSuccess;
}
hipError_t
hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
  *e = nullptr;
  return hipSuccess;
}
hipError_t
hipEventDestroy(hipEvent_t)
{
  return hipSuccess;
}
hipError_t
hipEventRecord(hipEvent_t, hipStream_t)
{
  return hipSuccess;
}

} // extern "C"

static void
check(int rc)
{
  if (rc != DG_OK)
    {
      std::fprintf(stderr, "%s\n", dg_last_error());
      std::exit(1);
    }
}

static int64_t
submit(dg_server *s, int degree, int cells)
{
  dg_serve_request r    = {};
  r.degree              = degree;
  r.cells_per_direction = cells;
  r.velocity[0]         = 1.;
  r.width               = 0.1;
  r.final_time          = 0.01;
  r.courant             = 0.3;
  int64_t id            = 0;
  check(dg_server_submit(s, &r, &id));
  return id;
}

static void
run_and_take(dg_server *s, const int64_t *ids, int n, size_t bytes)
{
  for (int left = n, f = 0; left > 0; left -= f)
    check(dg_server_step(s, 1, nullptr, nullptr, &f));
  void *dst = std::malloc(bytes);
  for (int i = 0; i < n; ++i)
    check(dg_server_take_result(s, ids[i], dst));
  std::free(dst);
}

int
main()
{
  // the larger request alone nearly fills the budget: three vectors of
  // 12^3 cells with 5^3 values and the mesh arrays
  const size_t  big    = size_t(8) * 12 * 12 * 12 * 125;
  const size_t  small  = size_t(8) * 8 * 8 * 8 * 64;
  const int64_t budget = 3 * big + 12 * 12 * 12 * 216 + (100 << 10);
  dg_server    *s      = nullptr;
  check(dg_server_create(budget, nullptr, &s));
  int64_t ids[4];
  for (int64_t &id : ids)
    id = submit(s, 3, 8);
  run_and_take(s, ids, 4, small);
  ids[0] = submit(s, 4, 12);
  run_and_take(s, ids, 1, big);
  const size_t most   = peak;
  const int    before = n_malloc;
  ids[0] = submit(s, 4, 12);
  run_and_take(s, ids, 1, big);
  const int again = n_malloc - before;
  check(dg_server_destroy(s));
  std::printf("%lld %zu %d %zu\n", (long long)budget, most, again, live);
  return 0;
}
