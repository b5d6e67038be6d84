/* host_build.h -- host-side scene preparation (spectra, flattening, BVHs). */
#ifndef CLV_HOST_BUILD_H
#define CLV_HOST_BUILD_H
#include <stdint.h>

#include <string>
#include <vector>

#include "../../include/clovers_hip.h"
#include "clv_layout.h"

namespace clv {

struct HostScene {
  std::vector<Bvh4Node> nodes;        /* root = nodes[0] */
  std::vector<float> prims;           /* float4 records, 4 floats per unit */
  std::vector<PrimInfo> prim_info;
  std::vector<Xform> xforms;
  std::vector<DevMaterial> materials;
  std::vector<float> spd;             /* n x 400 */
  int32_t background_spd = -1;
  std::vector<DevLight> lights;
  std::vector<DevLightNode> light_nodes;
  std::vector<float> light_weights;   /* per light leaf: 2^-depth */
  uint32_t light_root = LT_EMPTY;     /* child word of the tree root */
  clv_camera_init camera;
  uint32_t n_prims = 0;
  uint32_t bvh_depth = 0;
  uint32_t n_objects = 0;
  uint32_t n_media = 0;               /* constant media: their records end prims, media_units long */
  uint32_t media_units = 0;
  double build_ms = 0.0;
  /* built for the device builder: no nodes; prims holds the records in
   * primitive order (then the media), with each one's offset (float4 units)
   * and culling box */
  bool device_bvh = false;
  std::vector<uint32_t> prim_unit;
  std::vector<float> prim_box;        /* 8 floats per primitive: lo.xyz, 0, hi.xyz, 0 */
  float clo[3] = {0, 0, 0}, chi[3] = {0, 0, 0};  /* bounds of the box centres */
  float lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};    /* bounds of the boxes */
};

/* Build everything the device needs from the descriptor.  Returns a
 * clv_status; *err holds the detail on failure.  device_bvh: leave the scene
 * BVH to the device builder (records in primitive order, boxes, no nodes). */
int build_host_scene(const clv_scene_desc *desc, HostScene *out, std::string *err, bool device_bvh = false);

/* the f32 threshold below which a ConeLight of this spread (radians) is dark */
float cone_threshold(float spread_rad);

/* Offsets of a scene inside the context's device arena, in elements of each
 * array (prims and spd in float4 units / floats). */
struct ArenaBase {
  uint32_t nodes = 0, units = 0, info = 0, xforms = 0, mats = 0, spd = 0, lights = 0, lnodes = 0;
};

/* Rewrite every index of a built scene for placement at `b`: interior child
 * words, leaf record offsets, record xform and info indices, materials, SPD
 * offsets, light-tree words.  Fails if a leaf offset leaves 28 bits. */
int rebase_host_scene(HostScene *hs, const ArenaBase &b, std::string *err);

/* The wavefront passes of a batch (see plan_passes). */
struct PassPlan {
  std::vector<DevItem> items;       /* all passes, concatenated */
  std::vector<uint32_t> first;      /* per pass: first item (one more entry: the end) */
  std::vector<uint32_t> paths;      /* per pass: paths */
  std::vector<uint32_t> res;        /* per pass: resolve threads */
  std::vector<uint32_t> depth;      /* per pass: largest max_depth of its jobs */
  std::vector<uint8_t> train;       /* per pass: holds a training slice of a guided job */
  uint32_t max_paths = 0;
};

/* Split the jobs' samples into wavefront passes of about `target` paths: a
 * pass takes whole-sample slices (every pixel of a job, `samples` samples
 * each) from the unfinished jobs in turn, starting after the job that ended
 * the previous pass, until the target is reached; a job larger than the
 * target still gets one sample per pass.  A guided job's first `rounds`
 * slices hold at most `guided_cap` samples and mark their pass for a
 * training round.  With `warmup` those training slices are extra samples
 * (ITEM_WARMUP, stream indices from WARMUP_SAMPLE_BASE) ahead of the job's
 * own, which then all use the trained network.  Uses width, height, spp,
 * max_depth, guiding of `jobs`. */
void plan_passes(const std::vector<DevJob> &jobs, const std::vector<uint32_t> &sample_offset, uint32_t target,
                 uint32_t guided_cap, uint32_t rounds, bool warmup, PassPlan *pl);
/* join the passes behind the last training one, in order, into passes of at
 * most `target` paths (a pass already larger stays): no training round lies
 * between them, so no path changes */
void merge_passes(PassPlan *pl, uint32_t target);

/* Camera::new (camera.rs:59-99) for the given aspect ratio. */
DevCamera make_camera(const clv_camera_init &ci, float aspect);

/* wavelength_into_xyz (wavelength.rs:62-83) for lambda = 380..779: 400 x float4 (x, y, z, 0). */
void cie_xyz_table(float *out1600);

/* spectral_power (spectrum.rs:46-56): exposed for the spectral tests. */
float spectral_power(const float xyz[3], int lambda);

}  // namespace clv
#endif
