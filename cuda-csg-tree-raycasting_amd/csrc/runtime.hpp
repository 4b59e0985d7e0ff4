// Internals shared by the C ABI's translation units: the scene handle,
// error reporting, option parsing, job construction and per-stream device
// workspaces.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "csg.h"
#include "device.hpp"
#include "scene.hpp"

struct csg_scene {
  csgray::CSGTree tree;
  csgray::FlatScene flat;
  int device = 0;
  void* dmem = nullptr;
  size_t bytes = 0;
  csgray::DevScene dev{};
};

namespace csgray {
namespace rt {

// Records `msg` as the calling thread's last error and returns `s`.
csg_status Fail(csg_status s, const std::string& msg);
csg_status FailHip(hipError_t e, const char* what);

csg_status ParseOpts(const csg_render_opts* opts, LaunchConfig* cfg);
size_t SceneBytes(const csg_scene* s);

// Whether the tile kernel takes Union groups of the scene.
inline bool HasTileGroups(const csg_scene* s) { return s->dev.tileOps != s->dev.ivOps; }

// The scenes of one launch, as the choice of its kernels needs them.
struct LaunchScenes {
  int32_t maxOps, maxLeaves;
  bool inBoxes = false, groups = false;
  bool insideOut = false;  // boxes that do not hold their subtrees, as whole tiles and groups require
  // what the launch would lose by whole tiles, and what without them (us)
  double byTiles = 0, byLanes = 0;
  double chain = 0;       // of byTiles: the longest walk of a large tree in few tiles, beyond its time per lane
  int64_t largeWork = 0;  // tiles x operators of trees of kLaneLargeOps operators and more
  explicit LaunchScenes(int32_t least) : maxOps(least), maxLeaves(least) {}
  // A job of `tiles` 8x8 tiles (all samples).
  void Add(const csg_scene* s, int64_t tiles, Mode mode);
  // Whether the launch keeps the per-lane kernel, whatever its options.
  bool KeepsLanes(Mode mode) const;
};

// Validates one job and fills its device descriptor; `tileBase` is its first
// queue index within the launch.
csg_status BuildJob(const csg_scene* s, const csg_camera* cam, const csg_light* light, const csg_phong* phong,
                    int32_t width, int32_t height, const csg_outputs* out, const csg_render_opts* opts, int dev,
                    int64_t tileBase, Job* jb);

// The tile queue (five words, zero between launches) of (device, stream).
csg_status QueueFor(int dev, hipStream_t stream, uint32_t** out);

// The heavy-ray list of (device, stream).
csg_status HeavyFor(int dev, hipStream_t stream, uint2** out);

// Fills the tile kernel's and the cooperative kernel's fields of `p`
// (deferral off when the options say so or the cooperative kernel's state
// does not fit LDS).
void PrepareCoop(const LaunchConfig& cfg, const LaunchScenes& scenes, uint2* heavy, const LaunchShape& shape,
                 RenderParams* p);

// Copies a job table to the (device, stream) table buffer in stream order.
csg_status UploadJobs(int dev, hipStream_t stream, const Job* jobs, size_t n, const Job** out);

// Device bytes of one stream's workspace (queue, heavy-ray list with its
// resume area, job table for up to `maxJobs` jobs).
size_t StreamWorkspaceBytes(int32_t maxJobs);

// Frees the queue, heavy-ray list and job table of (device, stream); the
// caller has synchronised the stream and renders no more on it.
csg_status ReleaseStreamWorkspace(int dev, hipStream_t stream);

}  // namespace rt
}  // namespace csgray
