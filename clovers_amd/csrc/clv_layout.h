/*
 * clv_layout.h -- HBM data layout shared by the host builder and the HIP
 * kernels.  Plain structs, no HIP types, so both g++ and hipcc include it.
 *
 * Scene data (resident in HBM for the scene's lifetime):
 *   nodes      BVH4 nodes, 128 B each, 128-B aligned: child boxes as SoA
 *              (lo/hi per axis x 4 children) + 4 child words.
 *   prims      variable-size primitive records in float4 units:
 *                sphere 2 x float4 (32 B), moving sphere 3 x float4 (48 B:
 *                centre at time 0, radius, centre_1 - centre_0), quad and
 *                triangle 5 x float4 (80 B: q, u, v, plane d, unit normal,
 *                w = n / n.n), constant medium 3 x float4 with a
 *                sphere boundary or 32 x float4 with a box boundary (its six
 *                quad records; media are not in the BVH: each scene's media
 *                records follow its leaf records and every ray tests them
 *                after the tree); word .w of float4 #0 is the header
 *              (type | (xform+1) << 3), word .w of float4 #1 the primitive
 *              index into prim_info.
 *   prim_info  per primitive: material, reported id (object*8 + face).
 *   xforms     instance chains (RotateY/Translate), outermost op first.
 *   materials  per material: kind, SPD table offsets, scalar parameters.
 *   spd        n x 400 f32 spectral tables (index = lambda - 380).
 *   lights     the multiple-importance-sampling tree over priority objects:
 *              light records + a binary tree for sampling + leaf weights for
 *              the pdf (each leaf weighs 2^-depth, bvh/hitable_trait.rs:89-127).
 */
#ifndef CLV_LAYOUT_H
#define CLV_LAYOUT_H
#include <stdint.h>

#define CLV_LAMBDA_MIN 380
#define CLV_SPECTRUM 400

/* primitive types in record headers */
#define PT_SPHERE 0u
#define PT_QUAD 1u
#define PT_TRI 2u
#define PT_MSPHERE 3u
#define PT_MEDIUM 4u
#define PT_TYPE_MASK 7u   /* header bits of the type; the xform index + 1 sits above them */
#define PT_XF_SHIFT 3u

/* record sizes in float4 units */
#define PREC_SPHERE 2u
#define PREC_TRI 5u
#define PREC_QUAD 5u
#define PREC_MSPHERE 3u
/* record size by type as a nibble table: PT_SPHERE 2, PT_QUAD 5, PT_TRI 5, PT_MSPHERE 3
 * (a medium's size is in its record: see PREC_UNITS) */
#define PREC_TABLE 0x3552u
#define PREC_OF(type) ((PREC_TABLE >> ((type) << 2)) & 0xFu)

/* constant medium record (objects/constant_medium.rs):
 *   [-1/density, boundary kind, record units, header] [0, 0, 0, info]
 *   then the boundary: MED_SPHERE [centre, radius]; MED_BOX the six Boxy quads
 *   (boxy.rs:43-83) as quad records, in the reference's face order */
#define MED_SPHERE 0u
#define MED_BOX 1u
#define PREC_MED_SPHERE 3u
#define PREC_MED_BOX (2u + 6u * PREC_QUAD)
/* units of the record at rec (float4 units) whose header word is hdr; the
 * medium's size word is float4 #0 .z */
#define PREC_UNITS(hdr, size_word) \
  (((hdr) & PT_TYPE_MASK) == PT_MEDIUM ? (size_word) : PREC_OF((hdr) & PT_TYPE_MASK))

/* BVH4 child word: interior node index, or a leaf, or empty */
#define CHILD_LEAF 0x80000000u
#define CHILD_EMPTY 0xFFFFFFFFu
/* leaf: bit31 | count-1 (3 bits, <= 8 prims) << 28 | first record offset (float4 units, 28 bits) */
#define LEAF_MAX_PRIMS 8u
#define LEAF_OFFSET_MASK 0x0FFFFFFFu

typedef struct {
  float lo_x[4], hi_x[4], lo_y[4], hi_y[4], lo_z[4], hi_z[4];
  uint32_t child[4];
  uint32_t pad[4];
} Bvh4Node; /* 128 bytes */

typedef struct {
  uint32_t material;
  uint32_t report_id;    /* object_index * 8 + face */
} PrimInfo;

/* one instance op, outermost first */
#define XF_TRANSLATE 0u
#define XF_ROTATE_Y 1u
typedef struct {
  uint32_t kind;
  float a, b, c;         /* TRANSLATE: offset; ROTATE_Y: a = sin(theta), b = cos(theta) */
} XformOp;
typedef struct {
  uint32_t n_ops;
  uint32_t pad[3];
  XformOp ops[4];
} Xform;                 /* 80 bytes */

/* material classes used to sort hits into shading queues */
#define MC_MISS 0u
#define MC_LIGHT 1u
#define MC_LAMBERTIAN 2u
#define MC_METAL 3u
#define MC_GLASS 4u
#define MC_COUNT 5u

/* how a material's texture picks its SPD per hit */
#define TX_PLAIN 0u      /* one table: solid colour or illuminant */
#define TX_SPATIAL 1u    /* checker by world position: odd cells where sin(dx)sin(dy)sin(dz) < 0 */
#define TX_SURFACE 2u    /* checker by surface (u, v): odd cells where sin(du)sin(dv) < 0 */

typedef struct {
  uint32_t kind;         /* clv_material_kind */
  uint32_t mclass;       /* MC_* */
  int32_t albedo_spd;    /* offset of the reflectance SPD in spd[] (or -1); checkers: even cells */
  int32_t emit_spd;      /* offset of the emission SPD (or -1); checkers: even cells */
  float fuzz;            /* metal */
  float ior;             /* dielectric refractive index */
  float cauchy_a, cauchy_b;
  uint32_t thin_film;
  float film_ior, film_thickness;
  uint32_t tex;          /* TX_* of the albedo (Lambertian/Metal) or emission (lights) texture */
  int32_t odd_spd;       /* checkers: offset of the odd cells' SPD */
  float density_pi;      /* checkers: density * pi (the reference's f32 product) */
  float cone_cos;        /* ConeLight: c = -d.n / (|d| |n|) in [-1, 1] is outside the cone iff
                            c < cone_cos (the f32 threshold of acos(c) > spread in radians) */
  uint32_t cone;         /* 1: ConeLight */
} DevMaterial;           /* 64 bytes; Isotropic is kind CLV_MAT_ISOTROPIC in class MC_LAMBERTIAN */

/* light (MIS target) record: the reference's Quad/Triangle/Sphere params */
typedef struct {
  uint32_t type;         /* PT_* */
  uint32_t mat;          /* the object's material (arena index): emitters start light-traced training paths */
  uint32_t pad0[2];
  float q[4];            /* quad/tri: q, sphere: center */
  float u[4];            /* quad/tri: u; sphere: u[0] = radius */
  float v[4];
  float n[4];            /* unit normal, n[3] = d */
  float w[4];            /* w = n/(n.n), w[3] = area */
} DevLight;              /* 96 bytes */

/* light tree node for sampling: child word = node index | LT_LEAF | leaf index, or LT_EMPTY */
#define LT_LEAF 0x80000000u
#define LT_EMPTY 0xFFFFFFFFu
typedef struct {
  uint32_t child[2];
} DevLightNode;

typedef struct {
  float llc[3], horizontal[3], vertical[3], origin[3], u[3], v[3];
  float lens_radius;
  float pad;
} DevCamera;

/* per-job constants of a batch: one view of one scene */
typedef struct {
  DevCamera cam;
  uint32_t root;          /* BVH root node (arena index) */
  uint32_t light_root;    /* light-tree root word (arena indices) */
  uint32_t light_base;    /* the scene's MIS leaves: lights[light_base, +n_lights) */
  uint32_t n_lights;
  int32_t bg_spd;         /* background SPD offset in spd[] */
  uint32_t width, height;
  uint32_t max_depth;
  uint64_t seed;
  uint32_t pixel_base;    /* first accumulator pixel of the job */
  uint32_t spp;           /* samples per pixel of the whole job */
  uint32_t fp64;          /* accumulate in f64 */
  uint32_t guiding;        /* clv_guiding */
  float lo[3], hi[3];      /* scene box: guiding inputs are positions normalised to it */
  uint32_t media_off;      /* the scene's constant-medium records: prims[media_off ...], n_media of them */
  uint32_t n_media;
} DevJob;

/* one job's share of a wavefront pass: `samples` samples of every pixel */
typedef struct {
  uint32_t job;
  uint32_t path_base;     /* first path slot of the item */
  uint32_t pixels;        /* W*H of the job */
  uint32_t samples;       /* samples per pixel in this pass */
  uint32_t sample_base;   /* absolute index of the item's first sample */
  uint32_t res_base;      /* first resolve thread of the item (prefix sum of pixels) */
  uint32_t order;         /* pixel order of the item's slots within a sample: 0 row-major, 1 8x8 tiles */
  uint32_t flags;         /* ITEM_WARMUP: the samples train the guiding network only, the image never sees them */
} DevItem;
#define ITEM_WARMUP 1u
#define ITEM_FIRST 2u   /* holds the job's first samples */
#define ITEM_LAST 4u    /* holds the job's last samples */
/* warm-up samples take stream indices from here on, apart from any image sample */
#define WARMUP_SAMPLE_BASE 0x80000000u

#endif
