// Host-side session object: one reconstruction (volume, live-frame maps,
// model maps, pose state) with its own HIP stream.  The public opaque types
// dm_volume and dm_session both point at this object.
#pragma once
#include <hip/hip_runtime.h>
#include <string>
#include <vector>
#include "../../include/dynamap.h"
#include "../../include/dynamap_session.h"
#include "dm_internal.h"

namespace dm {

void set_error(const std::string &msg);
int hip_fail(hipError_t e, const char *what);

#define DM_HIP(call)                                 \
  do {                                               \
    hipError_t e_ = (call);                          \
    if (e_ != hipSuccess) return hip_fail(e_, #call); \
  } while (0)

// propagate a DM_* status
#define DM_TRY(x)                  \
  do {                             \
    int rc_ = (x);                 \
    if (rc_ != DM_OK) return rc_;  \
  } while (0)

struct Sess {
  dm_tsdf_props props{};
  dm_icp_props icp{};
  uint32_t max_rows = 0, max_cols = 0;
  DmView h{};                    // host copy of the view
  DmView *d_view = nullptr;      // device copy (one-entry table)
  int *d_active = nullptr;       // device {0}
  hipStream_t stream = nullptr;
  int device = 0;                // HIP device the state lives on (current at init)
  std::vector<void *> allocs;    // device allocations owned by the session
  float *d_depth = nullptr;      // frame staging
  uint8_t *d_rgb = nullptr;
  uint8_t *h_pinned = nullptr;   // pinned staging for host inputs
  size_t pinned_bytes = 0;
  size_t out_half = 0;           // bytes of one half of it, for results
  float *d_ray_depth = nullptr;  // raycast outputs for host readback
  uint8_t *d_ray_rgb = nullptr;
  float *d_pack = nullptr;       // packed maps for host readback (7 floats per pixel, allocated when a map is first asked for)
  hipEvent_t ev_out[2] = {nullptr, nullptr};
  float *d_depth_f = nullptr;    // bilateral-filtered depth for tracking (when enabled)
  int filt_r = 0;                // filter radius, 0 = off
  int icp_mfma = 0;              // ICP linearisation on the matrix cores (dm_session_set_icp_reduce)
  float filt_sd = 0.f, filt_ss = 0.f;
  size_t hbm_bytes = 0;          // device bytes owned
  int frames = 0;

  int init(const dm_tsdf_props &p, uint32_t rows, uint32_t cols);
  void release();
  template <class T> int dalloc(T **ptr, size_t count, bool zero = true);
  void push_view(const float *pose = nullptr);  // store h (and the frame pose) on the device, in stream order
  Launch launch() const;
  int set_sensor(const dm_sensor *s);
  int stage_depth(const float *host_depth);  // upload the frame through pinned memory; h.depth / h.rgb are set
  int stage_rgb(const uint8_t *host_rgb);    // by frame_from_host
  int frame_from_host(const float *host_depth, const uint8_t *host_rgb, const float *pose);
  int reserve_out(bool pack);  // pack: with d_pack
  struct Out { void *dst; const void *src; size_t bytes; };
  int read_out(const Out *out, int n);       // device results to host memory; waits
  int read_small(void *dst, const void *src, size_t bytes);  // up to 1 KiB; waits for the stream
};

// bytes of device memory a session with these parameters needs
size_t session_bytes(const dm_tsdf_props &p, uint32_t rows, uint32_t cols);
int validate_props(const dm_tsdf_props &p);

}  // namespace dm
