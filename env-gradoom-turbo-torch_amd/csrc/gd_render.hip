// MI355X (gfx950) batched software renderer + observation pipeline.
//
// One frame for N lanes runs as a short chain of kernels on the caller's stream:
//
//   lane_tables     1 block / lane            view basis, pitch centre, camera sector; distance bounds of every height
//                                             level, plane rows, row slopes
//   wall_setup      1 block / lane or 256 linedefs  FWallCoords span+depths, span ownership bounds, the linedef's
//                                             entry in the candidate list of every column it can own, and the
//                                             nearest blocking hit of every column (64-bit atomicMin)
//   strip_key/order 1 thread / 64-col strip   longest strip first (counting sort on the longest list); columns that see more than 64 linedefs
//   wall_select     1 wave / strip            portal traversal: which drawseg every column pass selects, one record each
//                   (the longest: 8 to 32)
//   wall_geometry   13 to 21 waves / lane            the linedefs those passes draw, as lines over the columns: every division of the drawing
//   wall_raster     1 to 8 waves / strip      the recorded passes drawn: projection, clips, tiers, planes, masked mid-textures
//   plane_shade     1 wave / 64 columns x 16 rows  flat texel + light for every pixel a plane of the wall pass shows,
//                                             the wall tiers' palette indices
//   flat_gap        8 or 16 waves / gap column     per-pixel plane rays (fine point raster) for the gap pixels, vertical repair
//   flat_rows, flat_span_select, flat_tail, flat_span_finish
//                                             visplane repair of the rows where a gap pixel stayed unresolved
//   flat_shade      1 wave / gap column       the gap pixels' flats
//   decal           320 threads / lane        bullet chips on the wall tiers they hit (frames that carry decals
//                                             also keep the depth of wall pixels: wall_raster<true>)
//   sprite_pixels   thread per view pixel     billboards, nearest visible one first, or blended far -> near
//   weapon_overlay, hud                       player weapon, muzzle flash and status bar patches
//   observe         1 thread / obs pixel      PLAYPAL + exact area pool + gray + 4-frame stack
//   expand_rgb      1 thread / pixel          PLAYPAL expansion for callers that want RGB24 frames
//
// All fixed-point arithmetic is int64 like the reference's Torch code; float32
// expressions are evaluated operation by operation (-ffp-contract=off) so that
// palette-index frames are bit-identical to the reference.  Citations name
// /root/reference/src/gradoom/engine.py unless stated otherwise.

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <new>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/gradoom_amd.h"
#include "gd_divide.h"
#include "gd_order.h"
#include "gd_internal.h"
#include "gd_rules.h"

thread_local std::string g_error;
int gd_fail(int code, const std::string &message) { g_error = message; return code; }

namespace {

typedef long long i64;
typedef unsigned long long u64;

#define SW 320
#define VH 208
#define CAND_MAX 64          // candidate linedefs a screen column keeps in its own slots
// A column whose ray can reach more than CAND_MAX linedefs (a long corridor seen end on) gets a slot in the chunk's spill
// pool, where strip_order_kernel lists all of them, up to SPILL_DEPTH.  The pool continues the candidate blocks with
// the same layout (entry k of a column lies k * 320 entries on), SPILL_DEPTH x 320 entries per pool block, so a
// spilled column differs from the others only in where its list starts and how long it may be.
#define SPILL_DEPTH 256
#define SPILL_SHIFT 12       // cand_count of a spilled column: entries | (pool slot + 1) << SPILL_SHIFT
static_assert(SPILL_DEPTH < (1 << SPILL_SHIFT), "a spilled column's count and its pool slot share a word");
#define SEG_COLS 64           // columns of a traversal segment; a wavefront takes 64 / SEG_COLS segments, of any lanes
#define SEGS_PER_LANE (SW / SEG_COLS)
#define GD_INF __builtin_inff()

// engine.py:42-51, 139-156
#define FIXED_UNIT 65536LL
#define UINT32_MASK 0xFFFFFFFFLL
#define FINE_ANGLES 8192
#define ANGLE_90 (1LL << 30)
#define FOCAL_X_FIXED (160LL * 65536LL)
#define Y_ASPECT_FIXED ((320LL * 65536LL * 240LL) / (200LL * 320LL))
#define FOCAL_Y_FIXED (160LL * Y_ASPECT_FIXED)
#define FLOOR_VISIBILITY_FIXED ((160LL * 65536LL * (8LL * 65536LL)) / FOCAL_Y_FIXED)
#define WALL_VISIBILITY_FIXED (((FOCAL_Y_FIXED * (320LL * 600LL) / (320LL * 240LL * 3LL)) * (8LL * 65536LL)) >> 16)
#define SPRITE_MIN_DEPTH_FIXED 8192LL

// candidate flags
#define CF_GEO 1
#define CF_PROJ 2
#define CF_LEDGE 4
#define CF_ALONG_HI 8   // along > 0.5: the ray is nearer the linedef's end vertex
#define CF_FF 16        // camera on the front side of the linedef (float32 test)
// facts of the linedef itself: a pass asks for them of every linedef it considers, and a load from the lane's records would be
// another trip to memory (0.9 GB of records for 4096 lanes) in the chain it waits for
#define CF_ENDS_HERE 32 // its clipped span ends at this column
#define CF_NARROW 64    // its clipped span is at most two columns wide
#define CF_SHORT 128    // at most 32 map units long
#define CF_SUBPIXEL 256 // two-sided, and its clipped span at most one column wide
#define CF_ONE_SIDED 512
#define CF_SECTOR0 4096   // one of its sides faces sector 0, which stands in where a column has none

// wall record flags
#define WF_HC 1        // owns at least one column after every span test
#define WF_SPLIT 2     // projects through BSP fragments (engine.py:11472-11545, 12310-12380)
#define WF_ANYGEO 8    // some column ray hits the segment
// the facts a candidate shows at every column, in its flags' places (eval_segment copies them)
#define WF_FF CF_FF             // front facing (float32 test of engine.py:11376-11381)
#define WF_NARROW CF_NARROW
#define WF_SHORT CF_SHORT
#define WF_SUBPIXEL CF_SUBPIXEL // two-sided and at most one column wide (engine.py:11589-11591)
#define WF_ONE_SIDED CF_ONE_SIDED
#define WF_SECTOR0 CF_SECTOR0
#define WF_SHOWN (WF_FF | WF_NARROW | WF_SHORT | WF_SUBPIXEL | WF_ONE_SIDED | WF_SECTOR0)
#define WF_END_SHIFT 16   // bits 16 and up: the column at which the clipped span ends, WF_END_NONE if that is not a column
#define WF_END_NONE 1023

struct LaneCtx {
    float x, y, view_z, pitch_offset, fsin, fcos;
    i64 view_x_fixed, view_y_fixed, vsin, vcos, center_fixed, flash_light;
    i64 upper_clip, lower_clip;   // OWallMost's view-frustum slopes at the top and bottom row (engine.py:12402-12413)
    int sector;
    int last_ceiling_row;         // rows 0 .. last_ceiling_row of the view look at ceilings, the rest at floors (-1: all floors)
};

struct WallRec {   // one linedef seen from one lane
    int tx0, tx1, ty0, ty1;  // view-space endpoints, start then end (engine.py:11173-11205)
    i64 dl, dr;              // clipped endpoint depths (engine.py:10835-10852)
    i64 sl, sr;              // clipped half-open screen span (engine.py:10825-10868); a rejected
                             // linedef keeps whatever its projection produced, hence 64 bits
    short pl, pr;            // span used for ray ownership (engine.py:11347-11427), within [0, 320]
    int flags;
};

// What the selection half of a column pass hands to the drawing half (wall_select_kernel -> wall_raster_kernel): the
// drawseg the pass selected and, where a geometric portal path continues behind a projected solid
// (engine.py:12969-13069), that path.  `bits` holds the PB_* flags of the selection (they fit 16 bits).
struct __align__(16) PassRec {
    unsigned short wall, render_current, bits, ps_path;
    short ps_other;
    unsigned short marks;     // REC_*
    float distance;
};
#define REC_SIDE1 1       // the pass draws the back side
#define REC_OWN_ROWS 2    // the pass draws from a sector that is not the one its side faces, or through a BSP fragment: its rows are not
                          // the linedef's lines but its own (Scratch::pass_rows, written by wall_geometry_kernel)
#define PASS_MAX 255  // most column passes recorded per screen column (the count is a byte).  A chunk keeps room for as many as the
                      // map has sectors (a column runs at most that many passes), at least 16, at most PASS_MAX: Scratch::pass_slots.
                      // A column that needs more sets STATUS_PASS_OVERFLOW.

// What the drawing half of the traversal asks of a linedef seen from one lane, as straight lines over the screen columns: every
// division of it (OWallMost's of its four heights, the wallscan light's) depends on the linedef alone, not on the column.
struct __align__(16) ColumnLine {    // base + x * step
    i64 base, step;
    __device__ __forceinline__ i64 at(int x) const { return (i64)((u64)base + (u64)(i64)x * (u64)step); }
};
// A height's row is clamp(line >> 16) (engine.py:12294-12605).  A height that the view frustum cuts, or that lies beyond it, bends: it
// then shows row 0 over the columns [top0, top1) and row 208 over [bottom0, bottom1) (but not at column `collapsed`), and in the
// columns outside the linedef's own screen span the line `outside`.
struct HeightBend {
    unsigned int top;      // top0 | top1 << 10 | (collapsed + 1) << 20
    unsigned int bottom;   // bottom0 | bottom1 << 10 | bends << 31
};
struct __align__(16) WallGeo {
    ColumnLine line[4];        // front ceiling, front floor, back floor, back ceiling
    HeightBend bend[4];
    ColumnLine visibility[2];  // wallscan light of side 0 and 1 (engine.py:11217-11291)
    int tx0, tx1, ty0, ty1;    // as in WallRec
    int span0, span1;          // the linedef's screen span within [0, 320] (empty: span0 == span1)
    int past_left, spare;      // does the span start right of column 0?
    ColumnLine outside[4];     // of heights that bend
};
struct __align__(16) MaskedGeo {   // the same of a linedef's masked mid-texture (engine.py:13424-13744): its upper and lower edge
    ColumnLine line[2];
    ColumnLine scale;              // the column's sprite scale
    ColumnLine outside[2];
    HeightBend bend[2];
};
// What a linedef's side adds that no camera changes
struct __align__(16) WallSide {
    int tex[3];              // mid, lower, upper
    short other, spare;      // the sector behind the side (-1 = none)
    float offset_y, contrast;// vertical texture offset; +16 on vertical linedefs, -16 on horizontal ones (engine.py:12853-12861)
    i64 offset_x, repeat;    // 16.16 texture offset and linedef length
    i64 spare2;
};

// What the selection asks about a linedef it has come to, whatever the camera: in one place, so that it waits for memory once.  A pass is a chain of
// loads that depend on one another, a trip to memory each: next to a table for sectors, one for vertices, one for neighbours, two for the bridges' ranges
// (and the neighbours' ray tests asked for one after the other, a bridge's linedefs by number and then by sectors, linedef 0 again in every pass that finds
// none) the launch for the longest strips takes 385 us instead of 433 at 4096 lanes of the 4000-linedef map, the other 788 instead of 800; 1024 lanes of the
// 2000-linedef map 232 instead of 248 and 191 instead of 202.
// A choice between two of its members is made between their values: written between the members themselves it is one between addresses, which kept the record in
// private memory, written and read back in every pass.  The stage at 4096 lanes of the 4000-linedef map 643 us that way, 577 now; 2048 lanes 445, 422; 256 lanes 147, 125;
// 1024 of the 2000-linedef map 192, 175.
struct __align__(16) WallLinks {
    unsigned sectors;        // front | back << 16 (0xFFFF: none)
    unsigned vertices;       // start | end << 16
    int neighbour[2];        // direct_neighbor_table's row
    unsigned slots;
    int solid[2];            // where its entries in the solid bridge lists start, by its start and by its end
    unsigned solid_counts;   // how many they are, start | end << 16
};
// A vertex's linedefs with their sectors (vertex_wall_idx and wall_sectors in one place)
struct VertexLink { int wall; unsigned sectors; };

struct RecSpan {   // what a ray test of one linedef needs (eval_segment), kept for every linedef of the map; the full record
                   // above exists only for the linedefs the camera can see at all
    short pl, pr;
    int flags;
};

struct __align__(8) Cand {      // one linedef with a finite ray distance at one column
    unsigned short flags, wall;   // in this order: the entry's bits are the key below
    float dist;
};
// (distance, linedef, flags) of a candidate as one unsigned number.  Listed distances are positive, so their bit patterns
// order as they do: the smallest key is the nearest candidate, the lowest linedef on ties, which is how every scan of the
// traversal breaks them (no column lists a linedef twice).  CAND_KEY_NONE, greater than any entry's, stands for "none".
#define CAND_KEY_NONE 0x7F800000FFFFFFFFULL
__device__ __forceinline__ u64 cand_key(const Cand &q) { return ((u64)__float_as_uint(q.dist) << 32) | ((u64)q.wall << 16) | (u64)q.flags; }
__device__ __forceinline__ Cand key_cand(u64 key) { Cand q; q.flags = (unsigned short)key; q.wall = (unsigned short)(key >> 16); q.dist = __uint_as_float((unsigned)(key >> 32)); return q; }
__device__ __forceinline__ float cand_key_distance(u64 key) { return __uint_as_float((unsigned)(key >> 32)); }
__device__ __forceinline__ int cand_key_wall(u64 key) { return key == CAND_KEY_NONE ? 0x7fffffff : (int)((unsigned)key >> 16); }
__device__ __forceinline__ int cand_key_flags(u64 key) { return key == CAND_KEY_NONE ? 0 : (int)((unsigned)key & 0xFFFFu); }

struct Eval {      // distances/along/geometric/projected/left-edge of one linedef at one column;
                   // CF_ALONG_HI in flags carries (along > 0.5), the only use the traversal makes of along
    float dist;
    int flags;
};

#define WALL_ONE_SIDED 1
#define WALL_SPLIT 2
#define WALL_SHORT 4     // at most 32 map units long
#define WALL_SECTOR0 8   // one of its sides faces sector 0
#define WALL_BLOCKING_SHIFT 4
struct DeviceMap {  // device copy of gd_map_desc (device pointers) + fixed tables
    gd_map_desc d;
    const i64 *fine_sine;     // [8192]
    const i64 *fine_tangent;  // [4096]
    const float *cosine_correction;  // [320] cos(native_ray_offsets), supplied by the host
    const float *inverse_cosine;     // [320] 1 / cosine_correction, correctly rounded
    float strip_reach_scale[SW / 64];// per 64-column strip: 1.001 / (its smallest cosine_correction), inf if not positive
    float strip_far_scale[SW / 64];  // per 64-column strip: 0.999 / (its largest cosine_correction), 0 if any is not positive
    float fine_inverse;              // 1 / fine_cell
    // Sectors grouped by plane level, floors (in floor_levels order) then ceilings: CSR over
    // floor_level_count + ceil_level_count rows into level_boxes, one padded bounding box
    // (x0, y0, x1, y1) per sector outside which no point tests inside that sector.
    const int *level_box_ofs;
    const float4 *level_boxes;
    const float4 *level_box;             // [levels] one box around all sectors of the level: no probe point outside it lands in one
    // The coarse grid repacked for the crossing test of flat selection: per cell its item range, per
    // item one 16-byte record, per item edge a copy of the linedef's endpoints, so that a test is
    // three dependent loads (range, record, edges) instead of six.
    const int2 *cell_range;              // [cells] first item, one past the last
    const int4 *cell_item;               // [items] sector | GRID_ALWAYS_INSIDE, floor level index | ceiling level
                                         // index << 8 (or -1 when not recorded), first edge, one past the last
    const float4 *cell_edge;             // [item edges] x1, y1, x2, y2
    const WallSide *wall_side;           // [W,2]
    const unsigned int *sprite_texels;   // [patches, spr_max_h, spr_max_w] texel | its post's first row << 8 | opaque << 16: one load instead of three
    const int *masked_slot;              // [W] number of the linedef among those with a mid-texture on a two-sided side, else -1
    int masked_count;                    // how many there are
    const WallLinks *wall_links;         // [W]
    const VertexLink *vertex_links;      // by vertex_wall_ofs
    const int *wall_facts;               // [W] WALL_*, and from bit WALL_BLOCKING_SHIFT on the linedef's position in blocking_walls plus one, 0 when it does not block
    const unsigned int *sector_level;    // [S] index of the floor in floor_levels | index of the ceiling in ceil_levels << 16;
                                         // null when some sector's height is missing from the level lists
};

struct Overlays {   // device copy of gd_overlay_desc; count 0 = layer not loaded
    gd_overlay_desc d;
};

struct Scratch {    // per-chunk working memory, sized at create
    LaneCtx *ctx;          // [L]
    WallRec *rec;          // [L,W] written for the linedefs wall_setup_kernel does not cull; never read for the others
    RecSpan *span;         // [L,W] every linedef
    WallGeo *geo;          // [L,W] the linedefs some column pass draws, a lane's from the start of its run on (wall_geometry_kernel)
    unsigned int *geo_slot;// [L,W] where in geo (written for those linedefs only)
    unsigned int *named;   // [L,(W+31)/32] a bit per linedef some column pass draws (cleared by lane_tables_kernel, set by wall_select_kernel)
    unsigned int *own_rows;// [L] bit k: strip k holds a pass with REC_OWN_ROWS (the same)
    int lane_stride;       // lanes of the chunk's planes
    MaskedGeo *masked_geo; // [L,masked_count] those whose masked mid-texture is some column's nearest
    u64 *masked_hit;       // [L,320] cand_key of the nearest candidate with a masked mid-texture on the side facing the camera and a
                           // projection that owns the column, CAND_KEY_NONE if none (engine.py:13436-13460)
    uint2 *pass_rows;      // [pass_slots,L,320] the eight projected rows of a pass whose record carries REC_OWN_ROWS (written for those only)
    WallRec *frag_rec;     // [L,split_count,fragment_slots] FWallCoords of the BSP fragments of split linedefs
    float *scene_depth;    // [L,208,320] depth of the wall tier or masked texture a pixel shows (engine.py:11553, 12700, 13740),
                           // kept only for frames that draw wall decals, else null; scene_depth_at() has the others
    Cand *cand;            // [L,CAND_MAX,320], eight bytes an entry (with sectors and vertices in it, sixteen, wall_setup_kernel took 455 us for 395), then the spill pool [spill_slots / 320, SPILL_DEPTH, 320]
    int *cand_count;       // [L,320] entries listed (beyond CAND_MAX: the column wanted more than its own slots hold), or for
                           // a column with a pool slot: entries in the pool | (slot + 1) << SPILL_SHIFT
    int *spill_columns;    // [spill_slots] the columns (lane * 320 + column) that were given pool slots, in slot order
    int *spill_count;      // [1] columns that asked for a slot (cleared by lane_tables_kernel, counted by note_length)
    unsigned spill_base;   // where the pool starts in `cand`, in entries
    int spill_slots;       // pool slots of this chunk (a multiple of 320)
    unsigned short *flat_sector;// [L,208,320]
    unsigned char *flat_flags;  // [L,208,320] bit0 unresolved
    int2 *gap_columns;     // [L*320] the screen columns that hold view pixels no wall tier, plane or masked texture covers (they
                           // show the flat pass's picture), of every lane, as one work list: lane << 9 | column, and the rows
                           // they lie in, first | one past the last << 8.  Listed by wall_raster_kernel.
    int *gap_column_count; // [1] its length (cleared by lane_tables_kernel)
    unsigned int *flat_tail; // [L,2,320] per screen half and column: the first resolved pixel below the half's noted rows, row << 16 | sector,
                           // all ones if the column was not looking for one or found none
    int *flat_span;        // [L,4] first / last row of the ceiling half, then of the floor half, that holds a shown
                           // pixel the flat pass could not resolve and whose repair reads its row (208, -1 = none):
                           // the rows the row repairs work on
    int *flat_spans;       // [L*2] the (lane << 1 | half) with such rows, as one work list
    int *flat_span_count;  // [1] its length (cleared by lane_tables_kernel)
    int *flat_rows;        // [L*208] the noted rows of every lane as one work list, entry = lane << 8 | row, and from the end of the chunk's
                           // lanes on backwards those below them, as far as their halves of the screen go
    int *flat_row_count;   // [2] their lengths (cleared by lane_tables_kernel, filled by flat_rows_kernel)
    int pass_slots;        // passes a column can record in this chunk
    // where pass `pass` of a column lies in the three planes below: the passes that most columns make lie close together
    __device__ __forceinline__ size_t pass_at(int pass, int local, int x) const { return ((size_t)pass * (size_t)lane_stride + (size_t)local) * SW + (size_t)x; }
    PassRec *pass_rec;     // [pass_slots,L,320] the drawsegs of each column's passes, in pass order
    float *pass_path_distance;  // [pass_slots,L,320] distance of the portal path of a pass that carries PB_PS_KEEPS (written for those only)
    unsigned char *pass_count;  // [L,320] passes recorded for the column: up to its last pass that draws or moves a clip
    unsigned int *meta;    // [L,208,320] filled | floor | plane_sector+1 | clip_wall+1
    unsigned char *masked_texel; // [L,208,320] palette indices of masked mid-textures, where no frame takes them (band_finish_kernel); null
                                 // unless the assembly in LDS was chosen
    unsigned char *frame;  // [L,240,320] when the caller wants no indexed output
    u64 *block_hit;        // [L,320] nearest blocking linedef of the column ray: float bits of the distance << 32 |
                           // slot in blocking_walls, all ones when no ray hits (engine.py:10534-10557)
    int *sprite_listed;    // [L] the lane's billboards that reach the view at all (sprite_list_kernel)
    int *lane_blends;      // [L] does some live billboard of the lane blend with the pixel below it (sprite_style other than -1)?
                           // (lane_tables_kernel)
    unsigned char *sprite_late; // [L, SW / SPRITE_COLUMNS, SPRITE_ROW_PARTS] did this work-group of the billboards' early launch leave pixels to the
                           // late one? (Written for lanes that blend.  In the memory of strip_order, which nothing reads once the walls are drawn:
                           // memory of its own would make a lane's share larger, and gd_render_static would refuse maps that it takes.)
    unsigned char *strip_key;  // [L*SEGS_PER_LANE] expected traversal length of each (lane, segment of SEG_COLS columns)
    int *strip_order;      // [L*SEGS_PER_LANE] segments, longest expected traversal first
    volatile unsigned char *status;   // [2] sticky flags in pinned host memory: a candidate list, a list of passes was cut short
    float *level_reach;    // [L, floor levels + ceiling levels] lower bound of the distance from the
                           // camera to any point inside a sector with that plane level
    float *level_far;      // [L, floor levels + ceiling levels] upper bound of that distance
    unsigned int *level_masks;  // [L, LEVEL_BUCKETS, level_mask_words]: the plane levels a flat probe can reach at all, by
                                // bucket of the probe's distance scale (see level_bucket)
    i64 *level_plane;      // [L, floor levels + ceiling levels, 2] plane height (16.16) and its visibility factor
    i64 *row_slope;        // [L, 208] plane distance per unit of plane height on each view row
    i64 *step_scale;       // [L, 3, 2, 16] per log2 texture size (widths, then heights): the flat texture step per
                           // column, the fraction at screen column 0, the camera's offset
};
#define PLANE_LEVELS 32    // the per-lane plane tables of level lists up to this long (each) are staged in LDS by the
                           // shading kernels; longer lists are read where lane_tables_kernel left them

#define META_FILLED 0x80000000u   // an opaque wall tier owns the pixel; its palette index sits in the low byte of the
                                  // plane sector field (plane shading, which writes every other view pixel, stores it)
#define META_FLOOR 0x40000000u    // the owning plane is a floor
// when a launch paints billboards: all of them at the end; those that need not wait for the flat pass's pixels; the others
#define SPRITES_ALL 0
#define SPRITES_EARLY 1
#define SPRITES_LATE 2
#define META_GAP_COVERED META_FLOOR   // in the word of a gap pixel (no tier, no plane, no masked texture: the bit above means nothing
                                  // there): a billboard was painted over it before the flat pass's pixels were, which flat_shade_kernel respects
#define META_MASKED 0x20000000u   // a masked mid-texture was drawn over the pixel
#define META_SECTOR_SHIFT 16
#define META_SECTOR_MASK 0x1FFFu  // plane sector + 1
#define META_WALL_MASK 0xFFFFu    // sprite-clip linedef + 1

// Does the view pixel with this word show the flat pass's picture: no wall tier, no plane, no masked texture?
__device__ __forceinline__ bool gap_pixel(unsigned int word) { return !(word & (META_FILLED | META_MASKED)) && ((word >> META_SECTOR_SHIFT) & META_SECTOR_MASK) == 0; }

#define STATUS_CAND_OVERFLOW 0
#define STATUS_PASS_OVERFLOW 1
__device__ __forceinline__ int named_words(const gd_map_desc *m) { return (m->wall_count + 31) / 32; }
#define STEP_TABLE 96   // int64 entries per lane of Scratch::step_scale

__device__ __forceinline__ i64 mul64(i64 a, i64 b) { return (i64)((u64)a * (u64)b); }
__device__ __forceinline__ i64 shl64(i64 a, int s) { return (i64)((u64)a << s); }
// a * b for a multiplier known to fit 32 unsigned bits: two 32-bit multiplies instead of three
__device__ __forceinline__ i64 mul64_u32(i64 a, unsigned b) { return (i64)((u64)a * (u64)b); }
// Bits 16..47 of a * b, all that `((a * b) >> 16) & 0xFFFFFFFF` ever looks at: the low words' full product, and of the
// two cross products only their low 16 bits, which 24-bit multiplies of the operands' low halves give at full rate.
__device__ __forceinline__ unsigned mul64_bits_16_47(i64 a, i64 b) {
    const unsigned al = (unsigned)a, ah = (unsigned)((u64)a >> 32), bl = (unsigned)b, bh = (unsigned)((u64)b >> 32);
    const u64 low = (u64)al * (u64)bl;
    const unsigned cross = __umul24(al & 0xFFFFu, bh & 0xFFFFu) + __umul24(ah & 0xFFFFu, bl & 0xFFFFu);
    return (unsigned)(low >> 16) + (cross << 16);
}
__device__ __forceinline__ i64 tdiv(i64 a, i64 b) { return truncated_quotient(a, b, [](double d) { return __builtin_amdgcn_rcp(d); }); }
// Lanes of one wavefront leave words in memory for one another: the hardware keeps a wavefront's loads and stores of one place in order, the compiler has to.
__device__ __forceinline__ void wave_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }
// Lanes of one wavefront leave words in LDS for one another: the order is the program's, the compiler has to keep it.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Smallest / largest value of the wavefront, by lane moves (all lanes executing; the result is uniform).
template <int CONTROL, int ROWS> __device__ __forceinline__ int wave_move(int other, int v) { return __builtin_amdgcn_update_dpp(other, v, CONTROL, ROWS, 0xF, false); }
__device__ __forceinline__ int wave_min(int v) {
    const int none = 0x7fffffff;
    v = min(v, wave_move<0x111, 0xF>(none, v)); v = min(v, wave_move<0x112, 0xF>(none, v));   // row_shr:1, 2, 4, 8: the last lane of
    v = min(v, wave_move<0x114, 0xF>(none, v)); v = min(v, wave_move<0x118, 0xF>(none, v));   // every sixteen holds their smallest
    v = min(v, wave_move<0x142, 0xA>(none, v)); v = min(v, wave_move<0x143, 0xC>(none, v));   // row_bcast:15, 31: lane 63 that of all
    return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_max(int v) { return -wave_min(-v); }
// Value of `v` in lane `lane` of the wavefront; `lane` must be the same in every active lane.
__device__ __forceinline__ int bcast(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float bcast(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }
__device__ __forceinline__ i64 clampi(i64 v, i64 lo, i64 hi) { return v < lo ? lo : (v > hi ? hi : v); }
__device__ __forceinline__ i64 max64(i64 a, i64 b) { return a > b ? a : b; }
__device__ __forceinline__ i64 min64(i64 a, i64 b) { return a < b ? a : b; }
__device__ __forceinline__ i64 round_to_i64(float v) { return (i64)rintf(v); }
__device__ __forceinline__ i64 f64_to_i64(double v) {
    // Torch's CPU cast (x86 cvttsd2si): out of range or NaN -> INT64_MIN
    if (!(v >= -9223372036854775808.0 && v < 9223372036854775808.0)) return (i64)0x8000000000000000ULL;
    return (i64)v;
}
__device__ __forceinline__ int ilog2(int v) { return 31 - __clz(v); }
__device__ __forceinline__ bool finitef(float v) { return fabsf(v) < GD_INF; }
__device__ __forceinline__ float tolerance_of(float d) { return fmaxf(fabsf(d) / 128.0f, 4.0f); }

// ---------------------------------------------------------------------------------------------
// map relations (engine.py:399-484, 1578-1612), answered from vertex ids and the vertex CSR
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ int link_sector(unsigned sectors, int side) { return (int)(short)(side ? sectors >> 16 : sectors & 0xFFFFu); }
__device__ __forceinline__ int link_vertex(unsigned vertices, int slot) { return (int)(slot ? vertices >> 16 : vertices & 0xFFFFu); }
struct MapView {
    const gd_map_desc *m;
    const WallLinks *walls;
    const VertexLink *vertex_links;
    // are a's and b's sectors the same two?
    static __device__ __forceinline__ bool same_pair(unsigned a, unsigned b) { return a == b || a == (b >> 16 | b << 16); }
    static __device__ __forceinline__ bool incident(unsigned sectors, int sector) { return link_sector(sectors, 0) == sector || link_sector(sectors, 1) == sector; }
    static __device__ __forceinline__ bool has_vertex(unsigned vertices, int v) { return link_vertex(vertices, 0) == v || link_vertex(vertices, 1) == v; }
    static __device__ __forceinline__ bool two_sided_distinct(unsigned sectors) {
        const int front = link_sector(sectors, 0), back = link_sector(sectors, 1);
        return front >= 0 && back >= 0 && front != back;
    }
    __device__ __forceinline__ bool opposing(int a, unsigned a_sectors, unsigned a_vertices, int b, unsigned b_sectors, unsigned b_vertices) const {
        if (!same_pair(a_sectors, b_sectors) || link_sector(a_sectors, 1) < 0 || link_sector(b_sectors, 1) < 0 ||
            has_vertex(b_vertices, link_vertex(a_vertices, 0)) || has_vertex(b_vertices, link_vertex(a_vertices, 1))) return false;
        const float4 wa = *reinterpret_cast<const float4 *>(m->walls + 4 * a), wb = *reinterpret_cast<const float4 *>(m->walls + 4 * b);
        float ax = wa.z - wa.x, ay = wa.w - wa.y, bx = wb.z - wb.x, by = wb.w - wb.y;
        float dot = ax * bx + ay * by;
        float cross = ax * by - ay * bx;
        return dot < 0 && fabsf(cross) < 1e-6f;
    }
    // the one linedef at `vertex` between the two sectors that `a` and `b` do not share, and its sectors
    __device__ bool triangle_bridge(int vertex, int a, unsigned a_sectors, int b, unsigned b_sectors, int *index, unsigned *sectors) const {
        *index = 0; *sectors = 0;
        if (!two_sided_distinct(a_sectors) || !two_sided_distinct(b_sectors)) return false;
        int a0 = link_sector(a_sectors, 0), a1 = link_sector(a_sectors, 1), b0 = link_sector(b_sectors, 0), b1 = link_sector(b_sectors, 1);
        int shared_count = (a0 == b0 || a0 == b1) + (a1 == b0 || a1 == b1);
        if (shared_count != 1) return false;
        int shared = (a0 == b0 || a0 == b1) ? a0 : a1;
        const unsigned between = (unsigned)((a0 == shared) ? a1 : a0) | (unsigned)((b0 == shared) ? b1 : b0) << 16;
        int found = -1, count = 0;
        const int first = m->vertex_wall_ofs[vertex], last = m->vertex_wall_ofs[vertex + 1];
        for (int k = first; k < last; k += 4) {      // a vertex has four linedefs or so: all of them at once
            VertexLink link[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) link[j] = vertex_links[min(k + j, last - 1)];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (k + j < last && link[j].wall != a && link[j].wall != b && same_pair(link[j].sectors, between)) { found = link[j].wall; *sectors = link[j].sectors; ++count; }
        }
        if (count != 1) return false;
        *index = found;
        return true;
    }
    __device__ bool portal_bridge(int slot, int path, unsigned path_sectors, unsigned path_vertices, int owner, unsigned owner_sectors, unsigned owner_vertices, int *index) const {
        *index = 0;
        if (owner == path) return false;
        const int v = link_vertex(path_vertices, slot);
        unsigned sectors;
        return has_vertex(owner_vertices, v) && triangle_bridge(v, path, path_sectors, owner, owner_sectors, index, &sectors);
    }
    __device__ bool sector_bridge(int vertex, int pending, unsigned pending_sectors, int path, unsigned path_sectors, int *index, unsigned *sectors) const {
        *index = 0; *sectors = 0;
        return path != pending && triangle_bridge(vertex, pending, pending_sectors, path, path_sectors, index, sectors);
    }
};

#define LDS_SECTORS 512
#define LDS_TEXTURES 224   // textures whose size bits are staged in LDS (a multiple of 32); later ones read the global arrays
#define GRID_ALWAYS_INSIDE (1 << 30)   // grid item flag: the whole cell lies inside the sector

// Even-odd parity of one sector's edge sub-list around a point (engine.py:9598-9612, 10994-11015).
__device__ __forceinline__ bool inside_edges(const gd_map_desc *m, int e0, int e1, float px, float py) {
    int crossings = 0;
    for (int k = e0; k < e1; ++k) {
        const float4 e = *reinterpret_cast<const float4 *>(m->walls + 4 * m->grid_item_edges[k]);
        float dy = e.w - e.y;
        float safe_dy = fabsf(dy) < 1e-6f ? 1.0f : dy;
        bool crosses = (e.y > py) != (e.w > py);
        float crossing_x = e.x + (py - e.y) * (e.z - e.x) / safe_dy;
        crossings += (crosses && px < crossing_x) ? 1 : 0;
    }
    return crossings & 1;
}

// inside_edges over the repacked edge copies, two edges per step
__device__ __forceinline__ bool inside_edge_copies(const float4 *edges, int e0, int e1, float px, float py) {
    int crossings = 0;
    for (int k = e0; k < e1; k += 2) {
        const float4 a = edges[k], b = edges[k + 1 < e1 ? k + 1 : k];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float4 e = j == 0 ? a : b;
            float dy = e.w - e.y;
            float safe_dy = fabsf(dy) < 1e-6f ? 1.0f : dy;
            bool crosses = (e.y > py) != (e.w > py);
            float crossing_x = e.x + (py - e.y) * (e.z - e.x) / safe_dy;
            crossings += (k + j < e1 && crosses && px < crossing_x) ? 1 : 0;
        }
    }
    return crossings & 1;
}

// Cell of the point grid, or -1 when no sector can contain the point.
__device__ __forceinline__ int grid_cell_of(const gd_map_desc *m, float px, float py) {
    float fx = floorf((px - m->grid_min_x) / m->grid_cell);
    float fy = floorf((py - m->grid_min_y) / m->grid_cell);
    if (!(fy >= 0.0f) || !(fy < (float)m->grid_ny) || !(fx < (float)m->grid_nx)) return -1;
    int ix = fx < 0.0f ? 0 : (int)fx;   // column 0 also stands for everything left of the grid
    if (!(fx == fx)) return -1;
    return (int)fy * m->grid_nx + ix;
}

// Fine raster entries (top two bits): a decided sector, empty, or undecided with / without the
// masks of plane levels that can win in the cell.
#define FINE_KIND(v) ((unsigned)(v) >> 30)
#define FINE_DECIDED 0u
#define FINE_EMPTY 1u
#define FINE_MIXED 2u
#define FINE_UNKNOWN 3u
#define FINE_MASK_LEVELS 15

// Fine raster lookup.  Points outside the raster (or not finite) report FINE_UNKNOWN with a
// negative cell, and the caller locates them with grid_cell_of.  The coarse cell of a point
// inside the raster is (iy >> 3) * grid_nx + (ix >> 3): grid_cell is 8 * fine_cell and both
// grids pad their cells far beyond the rounding of either index computation.
// (fx, fy) is the point in raster cell units; anything within a small fraction of a cell of the
// true position will do, because decided cells keep a margin of half a map unit.
__device__ __forceinline__ unsigned fine_lookup_cells(const gd_map_desc *m, float fx, float fy, int *coarse_cell) {
    int ix = (int)floorf(fx), iy = (int)floorf(fy);
    *coarse_cell = -1;
    if ((unsigned)ix >= (unsigned)m->fine_nx || (unsigned)iy >= (unsigned)m->fine_ny || !(fx == fx) || !(fy == fy)) return 0xC0000000u;
    *coarse_cell = (iy >> 3) * m->grid_nx + (ix >> 3);
    return m->fine_sector[iy * m->fine_nx + ix];
}
__device__ __forceinline__ unsigned fine_lookup(const gd_map_desc *m, float inv_cell, float px, float py, int *coarse_cell) {
    int ix = (int)floorf((px - m->grid_min_x) * inv_cell), iy = (int)floorf((py - m->grid_min_y) * inv_cell);
    *coarse_cell = -1;
    if ((unsigned)ix >= (unsigned)m->fine_nx || (unsigned)iy >= (unsigned)m->fine_ny || !(px == px) || !(py == py)) return 0xC0000000u;
    *coarse_cell = (iy >> 3) * m->grid_nx + (ix >> 3);
    return m->fine_sector[iy * m->fine_nx + ix];
}

// _sector_at (engine.py:9598-9617): first sector with odd parity, 0 when none
__device__ int sector_at(const gd_map_desc *m, float px, float py) {
    int cell;
    unsigned fine = fine_lookup(m, 1.0f / m->fine_cell, px, py, &cell);
    if (FINE_KIND(fine) == FINE_EMPTY) return 0;
    if (FINE_KIND(fine) == FINE_DECIDED) return (int)(fine & 0xFFFFu);
    if (cell < 0) cell = grid_cell_of(m, px, py);
    if (cell < 0) return 0;
    for (int it = m->grid_cell_ofs[cell]; it < m->grid_cell_ofs[cell + 1]; ++it) {
        int item = m->grid_item_sector[it];
        if ((item & GRID_ALWAYS_INSIDE) || inside_edges(m, m->grid_item_edge_ofs[it], m->grid_item_edge_ofs[it + 1], px, py))
            return item & ~GRID_ALWAYS_INSIDE;
    }
    return 0;
}

// A flat probe of plane level k lands at distance cd = h_k * g from the camera, h_k the level's plane height and
// g = 192 / |row - centre| / cos(column) the pixel's own scale, and can only hit a sector whose level is k if
// reach_k <= cd <= far_k (level_reach / level_far): that is, if g lies in [reach_k / h_k, far_k / h_k].  With a plane
// level per sector a pixel would test hundreds of such intervals to find the few that hold its g, so the lane keeps,
// for each of LEVEL_BUCKETS ranges of g (6.5 to the octave from g = 0.7 up, the first and last open-ended), a bit set
// of the levels whose interval reaches into the range, a bucket to spare on either side (far more than the rounding of
// the logarithm or of g can move anything).  A probe then visits only the levels of its bucket, in level order, and
// applies the exact test to those: the bit sets only spare it levels the exact test would reject as well.
#define LEVEL_BUCKETS 64
#define LEVEL_MASK_WORDS_MAX 32     // up to 1024 plane levels (floors and ceilings together); beyond that every level is visited,
#define LEVEL_MASK_MIN_LEVELS 64    // and so it is with few levels, where the bit sets cost more than they spare
__device__ __forceinline__ int level_mask_words(const gd_map_desc *m) {
    const int levels = m->floor_level_count + m->ceil_level_count;
    return levels > LEVEL_MASK_MIN_LEVELS && levels <= 32 * LEVEL_MASK_WORDS_MAX ? (levels + 31) / 32 : 0;
}
__device__ __forceinline__ int level_bucket(float g) {
    if (!(g > 0.0f)) return 0;
    const float b = floorf((__log2f(g) + 0.5f) * 6.5f);
    return b <= 0.0f ? 0 : (b >= (float)(LEVEL_BUCKETS - 1) ? LEVEL_BUCKETS - 1 : (int)b);
}

// The lane's view (engine.py:10648-10658, 2122-2133, 9622-9631, 12384-12391, 9619), but for last_ceiling_row.
__device__ __forceinline__ LaneCtx lane_view(const DeviceMap &dm, const gd_lanes_desc &lanes, int n) {
    const float BAM_TO_RADIANS = (float)(2.0 * 3.14159265358979323846 / 4294967296.0);
    LaneCtx c;
    c.x = lanes.x[n]; c.y = lanes.y[n]; c.view_z = lanes.view_z[n];
    float angle = lanes.angle[n];
    i64 pitch_bam = lanes.pitch_bam[n];
    c.flash_light = lanes.flash_light ? lanes.flash_light[n] : 0;
    i64 retained_bam = lanes.angle_bam[n];
    float visible_angle = (float)retained_bam * BAM_TO_RADIANS;
    i64 angle_bam = retained_bam;
    if (angle != visible_angle) {
        float two_pi = (float)(2.0 * 3.14159265358979323846);
        float r = fmodf(angle, two_pi);
        if (r != 0.0f && (r < 0.0f)) r += two_pi;   // torch.remainder with a positive divisor
        angle_bam = round_to_i64(r / BAM_TO_RADIANS) & UINT32_MASK;
    }
    i64 xf = lanes.x_fixed[n], yf = lanes.y_fixed[n];
    float visible_x = (float)xf / 65536.0f, visible_y = (float)yf / 65536.0f;
    c.view_x_fixed = (c.x != visible_x) ? round_to_i64(c.x * 65536.0f) : xf;
    c.view_y_fixed = (c.y != visible_y) ? round_to_i64(c.y * 65536.0f) : yf;
    int fine = (int)((angle_bam >> 19) & (FINE_ANGLES - 1));
    c.vsin = dm.fine_sine[fine];
    c.vcos = dm.fine_sine[(fine + FINE_ANGLES / 4) & (FINE_ANGLES - 1)];
    c.fsin = (float)c.vsin / 65536.0f;
    c.fcos = (float)c.vcos / 65536.0f;
    i64 tangent_index = clampi((ANGLE_90 - pitch_bam) >> 19, 0, FINE_ANGLES / 2 - 1);
    i64 tangent = dm.fine_tangent[tangent_index];
    c.center_fixed = (i64)(VH / 2) * FIXED_UNIT + ((FOCAL_Y_FIXED * tangent) >> 16);
    c.upper_clip = tdiv(shl64(-c.center_fixed, 16), FOCAL_Y_FIXED);
    c.lower_clip = tdiv(shl64((i64)VH * FIXED_UNIT - c.center_fixed, 16), FOCAL_Y_FIXED);
    c.pitch_offset = (float)((tangent * 12582912LL) >> 16) / 65536.0f;
    c.sector = sector_at(&dm.d, c.x, c.y);
    return c;
}

// A lane's view, by one thread of its block, while the others clear the lane's lists; then the tables for the flat kernels:
//  * per plane level, how far the camera is, at least, from every sector at that level: a flat
//    probe nearer than that cannot land in such a sector (engine.py:10981-11024 tests the point
//    against every sector; here the far ones are ruled out by their bounding boxes);
//  * per plane level, the fixed-point plane height and visibility factor (engine.py:10588-10600);
//  * per view row, the plane distance slope (engine.py:10917-10931);
//  * per log2 texture size, the per-column texture steps (engine.py:10895-10902).
// The last three only depend on (lane, level), (lane, row) and (lane, size), so dividing once
// here spares plane shading four 64-bit divisions per pixel.
__global__ void __launch_bounds__(256) lane_tables_kernel(DeviceMap dm, gd_lanes_desc lanes, int lane_base, int lane_count, Scratch sc) {
    const int local = blockIdx.x;
    const int floors = dm.d.floor_level_count, levels = floors + dm.d.ceil_level_count;
    if (local >= lane_count) return;
    __shared__ LaneCtx c;
    __shared__ unsigned int masks_lds[LEVEL_BUCKETS * LEVEL_MASK_WORDS_MAX];
    if (threadIdx.x == 0) c = lane_view(dm, lanes, lane_base + local);
    else if (threadIdx.x == 64) {
        int *span = sc.flat_span + (size_t)local * 4;
        span[0] = VH; span[1] = -1; span[2] = VH; span[3] = -1;
        if (local == 0) { *sc.flat_span_count = 0; sc.flat_row_count[0] = 0; sc.flat_row_count[1] = 0; *sc.gap_column_count = 0; *sc.spill_count = 0; }
    }
    // the lane's per-column lists start empty
    for (int x = threadIdx.x; x < SW; x += blockDim.x) { sc.cand_count[(size_t)local * SW + x] = 0; sc.block_hit[(size_t)local * SW + x] = ~0ULL; sc.masked_hit[(size_t)local * SW + x] = CAND_KEY_NONE; }
    for (int k = threadIdx.x; k < named_words(&dm.d); k += blockDim.x) sc.named[(size_t)local * named_words(&dm.d) + k] = 0u;
    if (threadIdx.x == 0) sc.own_rows[local] = 0u;
    {   // does a live billboard of the lane blend with what lies under it?
        bool blends = false;
        if (lanes.sprite_style && lanes.sprite_alive)
            for (int k = threadIdx.x; k < lanes.sprite_slots; k += blockDim.x) {
                const size_t at = (size_t)(lane_base + local) * lanes.sprite_slots + k;
                blends |= lanes.sprite_alive[at] != 0 && lanes.sprite_style[at] != -1;
            }
        const int any = __syncthreads_or(blends ? 1 : 0);
        if (threadIdx.x == 0) sc.lane_blends[local] = any;
    }
    const float cx = lanes.x[lane_base + local], cy = lanes.y[lane_base + local];
    const int mask_words = level_mask_words(&dm.d);
    for (int k = threadIdx.x; k < LEVEL_BUCKETS * mask_words; k += blockDim.x) masks_lds[k] = 0u;
    __syncthreads();
    {
        // rows 0 .. last_ceiling_row look at ceilings
        static_assert(VH <= 256, "lane_tables_kernel: a thread a row");
        const int ceiling_rows = __syncthreads_count((int)threadIdx.x < VH && !(((float)(int)threadIdx.x - (103.5f + c.pitch_offset)) > 0));   // flat_center()
        if (threadIdx.x == 0) { c.last_ceiling_row = ceiling_rows - 1; sc.ctx[local] = c; }
    }
    for (int l = threadIdx.x; l < levels; l += blockDim.x) {
        float reach = GD_INF, far = 0.0f;
        for (int k = dm.level_box_ofs[l]; k < dm.level_box_ofs[l + 1]; ++k) {
            const float4 box = dm.level_boxes[k];
            float dx = fmaxf(fmaxf(box.x - cx, cx - box.z), 0.0f), dy = fmaxf(fmaxf(box.y - cy, cy - box.w), 0.0f);
            reach = fminf(reach, sqrtf(dx * dx + dy * dy));
            dx = fmaxf(fabsf(box.x - cx), fabsf(box.z - cx)); dy = fmaxf(fabsf(box.y - cy), fabsf(box.w - cy));
            far = fmaxf(far, sqrtf(dx * dx + dy * dy));
        }
        // margin: the probe point is camera + unit ray * distance in float32, far inside 0.1%
        sc.level_reach[(size_t)local * levels + l] = reach * 0.999f - 0.5f;
        sc.level_far[(size_t)local * levels + l] = far * 1.001f + 0.5f;
        const float plane_height = l < floors ? (c.view_z - dm.d.floor_levels[l]) : (dm.d.ceil_levels[l - floors] - c.view_z);
        if (mask_words > 0 && plane_height > 0.0f && far >= reach) {      // a level at or beyond the eye shows no plane
            const float low = (reach * 0.999f - 0.5f) / plane_height, high = (far * 1.001f + 0.5f) / plane_height;
            const int first = max(level_bucket(low) - 1, 0), last = min(level_bucket(high) + 1, LEVEL_BUCKETS - 1);
            for (int b = first; b <= last; ++b) atomicOr(&masks_lds[b * mask_words + (l >> 5)], 1u << (l & 31));
        }
        const i64 plane_height_fixed = round_to_i64(plane_height * 65536.0f);
        sc.level_plane[((size_t)local * levels + l) * 2] = plane_height_fixed;
        sc.level_plane[((size_t)local * levels + l) * 2 + 1] = min64(tdiv(FLOOR_VISIBILITY_FIXED << 16, max64(plane_height_fixed, 1)), (1LL << 31) - 1);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < LEVEL_BUCKETS * mask_words; k += blockDim.x) sc.level_masks[(size_t)local * LEVEL_BUCKETS * mask_words + k] = masks_lds[k];
    for (int py = threadIdx.x; py < VH; py += blockDim.x) {
        i64 center_row = c.center_fixed >> 16;
        i64 pixel_y_fixed = (i64)py * FIXED_UNIT;
        i64 den = (py < center_row) ? (c.center_fixed - pixel_y_fixed - FIXED_UNIT / 2) : (pixel_y_fixed - c.center_fixed + FIXED_UNIT / 2);
        den = max64(den, 1);
        bool overflow = den <= (FOCAL_Y_FIXED >> 15);
        i64 yslope = tdiv(FOCAL_Y_FIXED << 16, den);
        sc.row_slope[(size_t)local * VH + py] = overflow ? (1LL << 31) - 1 : yslope;
    }
    for (int k = threadIdx.x; k < 32; k += blockDim.x) {
        const i64 basis = k < 16 ? c.vsin : c.vcos;
        const i64 step = tdiv(shl64(basis, 32 - (k & 15)), FOCAL_X_FIXED);
        i64 *entry = sc.step_scale + (size_t)local * STEP_TABLE;
        entry[k] = step;
        // the texture fraction of screen column 0 (column px is (px - 159) steps from the view axis), and the
        // camera's own offset in the texture, for the same log2 size
        entry[32 + k] = (shl64(k < 16 ? c.vcos : -c.vsin, 32 - (k & 15)) >> 16) - mul64(SW / 2 - 1, step);
        entry[64 + k] = shl64(k < 16 ? c.view_x_fixed : -c.view_y_fixed, 32 - (k & 15)) >> 16;
    }
}

__device__ __forceinline__ void ray_direction(const LaneCtx &c, int x, float *rx, float *ry) {
    // engine.py:10660-10670
    // (x - 160) / 160, correctly rounded: the reciprocal's product and one step (every column's quotient is the division's)
    const float across = (float)x - 160.0f, inverse = 1.0f / 160.0f, near = across * inverse;
    const float col = __builtin_fmaf(__builtin_fmaf(-160.0f, near, across), inverse, near);
    *rx = c.fcos + c.fsin * col;
    *ry = c.fsin - c.fcos * col;
}

// distances / along / geometric / projected / left-edge of one linedef at one column
// (engine.py:11317-11331, 11440-11460)
__device__ __forceinline__ Eval eval_segment(const float4 wl, int rec_flags, int rec_pl, int rec_pr, const LaneCtx &c, int x, float rx, float ry) {
    float segx = wl.z - wl.x, segy = wl.w - wl.y;
    float offx = wl.x - c.x, offy = wl.y - c.y;
    float den = rx * segy - ry * segx;
    bool ok = fabsf(den) >= 1e-6f;
    float safe = ok ? den : 1.0f;
    float d = (offx * segy - offy * segx) / safe;
    float a = (offx * ry - offy * rx) / safe;
    bool g = ok && (d > 0) && (a >= 0) && (a <= 1);
    bool screen_valid = (rec_flags & WF_HC) && (x >= rec_pl) && (x < rec_pr);
    bool p = ok && (d > 0) && screen_valid;
    bool valid = (rec_flags & WF_ONE_SIDED) ? (p && (rec_flags & WF_FF)) : (g || p);
    Eval out;
    out.dist = valid ? d : GD_INF;
    out.flags = (g ? CF_GEO : 0) | (p ? CF_PROJ : 0) | ((x == rec_pl) ? CF_LEDGE : 0) | ((a > 0.5f) ? CF_ALONG_HI : 0) |
                (((rec_flags >> WF_END_SHIFT) == x) ? CF_ENDS_HERE : 0) | (rec_flags & WF_SHOWN);
    return out;
}

__device__ __forceinline__ Eval eval_wall(const gd_map_desc *m, const LaneCtx &c, const RecSpan *spans, int x, int w, float rx, float ry) {
    const float4 wl = *reinterpret_cast<const float4 *>(m->walls + 4 * w);
    const RecSpan r = spans[w];
    return eval_segment(wl, r.flags, r.pl, r.pr, c, x, rx, ry);
}

// ---------------------------------------------------------------------------------------------
// wall_setup: engine.py:10747-10869 (FWallCoords) and the per-linedef half of 11304-11451
// ---------------------------------------------------------------------------------------------
// FWallCoords of one fixed-point segment seen from one lane (engine.py:10747-10869): view-space
// endpoints, clipped half-open screen span and clipped endpoint depths.
// `endpoint_quotient`, when asked for, receives tx * center / ty (ty == 0 counted as 1) of the linedef's two endpoints
// in map order: the projections below divide exactly these, whichever endpoint the facing puts first.
__device__ __forceinline__ void wall_coords(const LaneCtx &c, const int *wf, WallRec &r, i64 *endpoint_quotient = nullptr) {
    i64 rx0 = (i64)wf[0] - c.view_x_fixed, ry0 = (i64)wf[1] - c.view_y_fixed;
    i64 rx1 = (i64)wf[2] - c.view_x_fixed, ry1 = (i64)wf[3] - c.view_y_fixed;
    i64 tx0 = (rx0 * c.vsin - ry0 * c.vcos) >> 20, ty0 = (rx0 * c.vcos + ry0 * c.vsin) >> 20;
    i64 tx1v = (rx1 * c.vsin - ry1 * c.vcos) >> 20, ty1v = (rx1 * c.vcos + ry1 * c.vsin) >> 20;
    i64 vx = (i64)wf[2] - wf[0], vy = (i64)wf[3] - wf[1];
    i64 fx = c.view_x_fixed - wf[0], fy = c.view_y_fixed - wf[1];
    bool front = (vx * fy - vy * fx) < 0;
    i64 tx1 = front ? tx0 : tx1v, tx2 = front ? tx1v : tx0;
    i64 ty1 = front ? ty0 : ty1v, ty2 = front ? ty1v : ty0;
    const i64 center = 160 * FIXED_UNIT;
    const i64 quotient0 = tdiv(tx0 * center, ty0 == 0 ? 1 : ty0), quotient1 = tdiv(tx1v * center, ty1v == 0 ? 1 : ty1v);
    if (endpoint_quotient) { endpoint_quotient[0] = quotient0; endpoint_quotient[1] = quotient1; }
    i64 left_projected = ((center + (front ? quotient0 : quotient1)) >> 16) + (tx1 >= 0);
    if (tx1 >= 0) left_projected = min64(left_projected, SW);
    i64 right_projected = ((center + (front ? quotient1 : quotient0)) >> 16) + (tx2 >= 0);
    if (tx2 >= 0) right_projected = min64(right_projected, SW);
    i64 left_den = tx1 - tx2 - ty2 + ty1, right_den = ty2 - ty1 - tx2 + tx1;
    i64 safe_left_den = left_den == 0 ? 1 : left_den, safe_right_den = right_den == 0 ? 1 : right_den;
    bool left_inside = tx1 >= -ty1, right_inside = tx2 <= ty2;
    i64 sl = left_inside ? left_projected : 0;
    i64 sr = right_inside ? right_projected : SW;
    i64 dl = left_inside ? ty1 : ty1 + tdiv((ty2 - ty1) * (tx1 + ty1), safe_left_den);
    i64 dr = right_inside ? ty2 : ty1 + tdiv((ty2 - ty1) * (tx1 - ty1), safe_right_den);
    bool invalid_left = (left_inside ? ((tx1 > ty1) || (ty1 == 0)) : ((tx2 < -ty2) || (left_den == 0))) || (dl < 32);
    bool invalid_right = (right_inside ? ((tx2 < -ty2) || (ty2 == 0)) : ((tx1 > ty1) || (right_den == 0))) || (dr < 32);
    bool invalid = invalid_left || invalid_right || (sr <= sl);
    if (invalid) sr = sl;
    r.tx0 = (int)tx0; r.tx1 = (int)tx1v; r.ty0 = (int)ty0; r.ty1 = (int)ty1v;
    r.dl = dl; r.dr = dr; r.sl = sl; r.sr = sr;
}

// Every fragment of every split linedef of one lane (engine.py:11472-11500).
__global__ void fragment_setup_kernel(DeviceMap dm, int lane_count, Scratch sc) {
    const gd_map_desc *m = &dm.d;
    const int per_lane = m->split_count * m->fragment_slots;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int local = blockIdx.y;
    if (local >= lane_count || k >= per_lane) return;
    WallRec r;
    wall_coords(sc.ctx[local], m->split_fragments_fixed + 4 * (size_t)k, r);
    r.pl = 0; r.pr = 0; r.flags = 0;
    sc.frag_rec[(size_t)local * per_lane + k] = r;
}

// A column that was offered more entries than its own slots hold asks for a slot in the spill pool.  With the pool
// used up the column keeps its first CAND_MAX entries and the renderer's status says so.
__device__ __forceinline__ void request_spill_slot(const Scratch &sc, int column) {
    const int slot = atomicAdd(sc.spill_count, 1);
    if (slot < sc.spill_slots) sc.spill_columns[slot] = column;
    else sc.status[STATUS_CAND_OVERFLOW] = 1;
}

// The expected traversal length of a strip, from its columns' counts, a lane a column (see strip_order_kernel); columns that see too
// many linedefs ask for a slot of the spill pool.
__device__ __forceinline__ void note_length(const Scratch &sc, int local, int x, int length) {
    static_assert(SEG_COLS == 64, "note_length: a strip a wavefront");
    if (length > CAND_MAX) { request_spill_slot(sc, local * SW + x); length = CAND_MAX; }
    length = wave_max(length);
    if ((x & (SEG_COLS - 1)) == 0) sc.strip_key[local * SEGS_PER_LANE + x / SEG_COLS] = (unsigned char)length;   // at most CAND_MAX
}

// One thread owns one linedef for the per-linedef arithmetic; its columns are looked at by the whole wavefront together, since
// linedefs reach from none of them to all 320.  A linedef has a window of columns its rays or its owned span can lie in, so one
// look at each of them says where its rays hit it, which gives the span it owns, which says where it is a candidate.  Windows of up
// to 8, 16 and 32 columns share a turn, as many linedefs as fit, a wider one has the wavefront to itself.  What a turn asks of its
// linedefs lies in LDS, and so do the lists of linedefs by width.
//
// Three quarters of a map's linedefs lie wholly behind the camera or wholly to one side of its view: no
// column ray can hit such a linedef and FWallCoords rejects it, so nothing of it is ever looked at beyond
// the ray-test facts of RecSpan (no owned span).  A block first sorts its linedefs into those and the
// rest, and only the rest are shared out over its wavefronts.
// Bound by its vector instructions, then by the latency of a turn's steps.  4096 lanes on the 4000-linedef map: 0.61 ms with two looks a
// column (one for the hits, one for the candidates), parameters by lane exchange and counts by atomics in device memory, 0.53 with one
// look and LDS parameters, 0.45 with counts in LDS; 16 lanes on the 320-linedef map 0.040 -> 0.019.
#define SETUP_WHOLE_THREADS 512
#define SETUP_WALLS_MAX 4096      // linedefs sorted at a time
struct SetupWall {                // a linedef as the columns' look at it asks for it
    float segx, segy, offx, offy;
    float numer;                  // of the ray distance
    int window;                   // first column | one past the last << 16
    int facts;                    // WF_* but for WF_HC and WF_ANYGEO, and SETUP_*
    int ends;                     // screen column of the left endpoint | of the right one << 9 | their visibility << 18, 19
    int wall;
    int blocking;                 // its position in blocking_walls, -1
};
#define SETUP_MASKED 0x400        // free bits of the WF_* word: a mid-texture on the side facing the camera
#define SETUP_SPANS 0x800         // FWallCoords' span is not empty
// The span a linedef owns (engine.py:11347-11427), within [0, 320]: first column | one past the last << 16, bit 31 when it owns any.
__device__ __forceinline__ int setup_owned(int facts, int ends, bool any, int first, int last) {
    const int left = ends & 511, right = (ends >> 9) & 511;
    const bool left_visible = (ends >> 18) & 1, right_visible = (ends >> 19) & 1;
    const bool both = left_visible && right_visible;
    const int from = both || (any && left_visible) ? left : first, to = both || (any && right_visible) ? right : last + 1;
    const bool owns = (both ? to > from : any) && (facts & SETUP_SPANS);
    return from | (to << 16) | (owns ? (int)0x80000000u : 0);
}
// WHOLE: one work-group goes over all linedefs of a lane, SETUP_WALLS_MAX at a time, and keeps what its columns count in LDS; else the
// linedefs of a lane are dealt out, SETUP_THREADS a work-group, and they count in device memory.
template <bool WHOLE>
__global__ void __launch_bounds__(WHOLE ? SETUP_WHOLE_THREADS : SETUP_THREADS) __attribute__((amdgpu_waves_per_eu(6, 6))) wall_setup_kernel(DeviceMap dm, int lane_count, Scratch sc) {
    const gd_map_desc *m = &dm.d;
    constexpr int THREADS = WHOLE ? SETUP_WHOLE_THREADS : SETUP_THREADS, WAVES = THREADS / 64, ROUND = WHOLE ? SETUP_WALLS_MAX : SETUP_THREADS;
    __shared__ unsigned short alive_list[ROUND];
    __shared__ int alive_count;
    __shared__ __align__(16) SetupWall walls_lds[WAVES][64];
    __shared__ int hits_lds[WAVES][64];                  // per linedef: first column a ray hits it at | one past the last << 16
    __shared__ unsigned char by_width[WAVES][3][64];     // the linedefs with windows of up to 8, 16, 32 columns
    __shared__ float wide_lds[WAVES][SW];                // a wide window's looks: the ray distance, negative where the ray is nearer the end, 0 for none
    __shared__ u64 wide_hits[WAVES][SW / 64];            // and the rays that hit, a word a turn
    __shared__ u64 block_lds[WHOLE ? SW : 1], masked_lds[WHOLE ? SW : 1];
    __shared__ int count_lds[WHOLE ? SW : 1];
    // ray_direction of every column, and of some that are looked at in vain: worked out at every look, ten instructions of some ninety, the kernel takes
    // 400 us for 386 (4096 lanes on the 4000-linedef map), 98 for 93 (1024 on the 2000-linedef map)
    __shared__ float2 rays_lds[SW + 64];
    const int slot = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int local = blockIdx.y;
    if (local >= lane_count) return;          // uniform over the block
    const LaneCtx &c = sc.ctx[local];
    u64 *block_hits = WHOLE ? block_lds : sc.block_hit + (size_t)local * SW, *masked_hits = WHOLE ? masked_lds : sc.masked_hit + (size_t)local * SW;
    int *counts = WHOLE ? count_lds : sc.cand_count + (size_t)local * SW;
    Cand *list = sc.cand + (size_t)local * CAND_MAX * SW;
    for (int x = threadIdx.x; x < SW + 64; x += THREADS) ray_direction(c, x, &rays_lds[x].x, &rays_lds[x].y);
    if (WHOLE) for (int x = threadIdx.x; x < SW; x += THREADS) { block_lds[x] = ~0ULL; masked_lds[x] = CAND_KEY_NONE; count_lds[x] = 0; }
    for (int round0 = WHOLE ? 0 : blockIdx.x * ROUND; round0 < (WHOLE ? m->wall_count : (int)(blockIdx.x + 1) * ROUND); round0 += ROUND) {
    __syncthreads();                                     // nobody reads the list of the round before any more
    if (threadIdx.x == 0) alive_count = 0;
    __syncthreads();
    for (int k = threadIdx.x; k < ROUND; k += THREADS) {
        const int w = round0 + k;
        bool kept = false;
        if (w < m->wall_count) {
            const float4 wl = *reinterpret_cast<const float4 *>(m->walls + 4 * w);
            const float ax = wl.x - c.x, ay = wl.y - c.y, bx = wl.z - c.x, by = wl.w - c.y;
            // forward and rightward view coordinates of both endpoints; a column ray is forward + col * right, |col| <= 1
            const float f0 = ax * c.fcos + ay * c.fsin, r0 = ax * c.fsin - ay * c.fcos;
            const float f1 = bx * c.fcos + by * c.fsin, r1 = bx * c.fsin - by * c.fcos;
            // wholly in one of the half planes behind the camera, right of the right view edge, left of the left one (a map
            // unit to spare, far more than float32 and 16.16 coordinates can disagree): no ray reaches it, FWallCoords finds
            // no span.  Linedef 0 and the first blocking linedef stand in where a scan finds nothing, and are always kept.
            const bool unseen = (f0 < -1.0f && f1 < -1.0f) || (r0 > f0 + 1.0f && r1 > f1 + 1.0f) || (r0 < -f0 - 1.0f && r1 < -f1 - 1.0f);
            kept = !unseen || w == 0 || (m->blocking_count > 0 && w == m->blocking_walls[0]);
            if (!kept) {
                const float vfx = c.x - wl.x, vfy = c.y - wl.y;
                const bool ff = ((wl.z - wl.x) * vfy - (wl.w - wl.y) * vfx) < 0;
                RecSpan span;
                span.pl = 0; span.pr = 0;
                // an unseen linedef has an empty span (sr == sl), so a two-sided one counts as at most one column wide
                const int facts = dm.wall_facts[w];
                span.flags = (ff ? WF_FF : 0) | ((facts & WALL_ONE_SIDED) ? WF_ONE_SIDED : WF_SUBPIXEL) | ((facts & WALL_SPLIT) ? WF_SPLIT : 0) |
                             WF_NARROW | ((facts & WALL_SHORT) ? WF_SHORT : 0) | ((facts & WALL_SECTOR0) ? WF_SECTOR0 : 0) | (WF_END_NONE << WF_END_SHIFT);
                sc.span[(size_t)local * m->wall_count + w] = span;
            }
        }
        const u64 keeps = __ballot(kept);
        int base = 0;
        if (slot == 0 && keeps) base = atomicAdd(&alive_count, __popcll(keeps));
        base = __builtin_amdgcn_readfirstlane(base);
        if (kept) alive_list[base + __popcll(keeps & ((1ULL << slot) - 1))] = (unsigned short)w;
    }
    __syncthreads();
    const int alive = alive_count;
    // the kept linedefs go to the wavefronts in equal shares, of at most 64
    const int shares = WHOLE ? (alive + 64 * WAVES - 1) / (64 * WAVES) * WAVES : WAVES;
    const int each = max((alive + shares - 1) / max(shares, 1), 8);
    for (int first_alive = wave * each; first_alive < alive; first_alive += WAVES * each) {
        const bool live = slot < each && first_alive + slot < alive;   // the other lanes help with the columns
        const int w = live ? alive_list[first_alive + slot] : 0;
        WallRec r;
        i64 endpoint_quotient[2];
        wall_coords(c, m->walls_fixed + 4 * w, r, endpoint_quotient);
        // Ray x segment: the columns whose ray hits the segment (engine.py:11323-11348).
        // A ray of column parameter col = (x-160)/160 is forward + col*right; an endpoint with view
        // coordinates (f, r) lies on it when r = col*f.  The float test below can only pass where the
        // two endpoints are not both clearly (> half a map unit) on one side of the ray, so for a
        // segment wholly in front of the camera only the columns between its endpoint columns
        // (padded) are examined; segments reaching behind the camera get the full scan.
        const float4 wl = *reinterpret_cast<const float4 *>(m->walls + 4 * w);
        const float segx = wl.z - wl.x, segy = wl.w - wl.y;
        const float offx = wl.x - c.x, offy = wl.y - c.y;
        int lo = 0, hi = SW;
        {
            const float e1x = offx + segx, e1y = offy + segy;
            const float f0 = offx * c.fcos + offy * c.fsin, r0 = offx * c.fsin - offy * c.fcos;
            const float f1 = e1x * c.fcos + e1y * c.fsin, r1 = e1x * c.fsin - e1y * c.fcos;
            if (f0 > 1.0f && f1 > 1.0f) {
                const float c0 = r0 / f0, c1 = r1 / f1, p0 = 0.5f / f0, p1 = 0.5f / f1;
                const float left = fminf(c0 - p0, c1 - p1), right = fmaxf(c0 + p0, c1 + p1);
                const float xlo = floorf(160.0f + 160.0f * left) - 1.0f, xhi = ceilf(160.0f + 160.0f * right) + 1.0f;
                lo = xlo < 0.0f ? 0 : (xlo > 320.0f ? 320 : (int)xlo);
                hi = (xhi > 319.0f ? 319 : (xhi < -1.0f ? -1 : (int)xhi)) + 1;
            } else if (f0 < -1.0f && f1 < -1.0f) {
                lo = SW; hi = 0;   // wholly behind the camera: no ray reaches it
            }
        }
        const bool ff = (segx * (c.y - wl.y) - segy * (c.x - wl.x)) < 0;
        int ends = 0;
        bool visible[2];
        {   // the endpoints' screen columns: tx * center / ty, as wall_coords divided it
            const i64 tx[2] = {r.tx0, r.tx1}, ty[2] = {r.ty0, r.ty1};
            int column[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const i64 col = ((160 * FIXED_UNIT + endpoint_quotient[e]) >> 16) + (tx[e] >= 0);
                visible[e] = (ty[e] > 0) && (tx[e] >= -ty[e]) && (tx[e] <= ty[e]) && (col >= 0) && (col <= SW);
                column[e] = visible[e] ? (int)col : 0;
            }
            // the owned span begins at the start of a linedef that faces the camera, at the end of one that does not
            ends = ff ? (column[0] | (column[1] << 9) | (visible[0] ? 1 << 18 : 0) | (visible[1] ? 1 << 19 : 0))
                      : (column[1] | (column[0] << 9) | (visible[1] ? 1 << 18 : 0) | (visible[0] ? 1 << 19 : 0));
        }
        // the window: where rays can hit, and the ends of what the linedef can own
        const bool scans = lo < hi;
        int window0 = scans ? lo : SW, window1 = scans ? hi : 0;
        if (ends & (1 << 18)) window0 = min(window0, ends & 511);
        if (ends & (1 << 19)) window1 = max(window1, (ends >> 9) & 511);
        const int known = dm.wall_facts[w];
        const bool os = known & WALL_ONE_SIDED;
        const i64 span = r.sr - r.sl;
        const int facts = (ff ? WF_FF : 0) | ((span <= 1 && !os) ? WF_SUBPIXEL : 0) | ((known & WALL_SPLIT) ? WF_SPLIT : 0) | (span <= 2 ? WF_NARROW : 0) |
                          ((known & WALL_SHORT) ? WF_SHORT : 0) | ((r.sr >= 0 && r.sr < SW ? (int)r.sr : WF_END_NONE) << WF_END_SHIFT) |
                          (os ? WF_ONE_SIDED : 0) | ((known & WALL_SECTOR0) ? WF_SECTOR0 : 0) | (!os && m->side_tex[(w * 2 + (ff ? 0 : 1)) * 3] >= 0 ? SETUP_MASKED : 0) | (span > 0 ? SETUP_SPANS : 0);
        {
            SetupWall mine;
            mine.segx = segx; mine.segy = segy; mine.offx = offx; mine.offy = offy;
            mine.numer = offx * segy - offy * segx;
            mine.window = window0 | (window1 << 16);
            mine.facts = facts; mine.ends = ends;
            mine.wall = w; mine.blocking = (known >> WALL_BLOCKING_SHIFT) - 1;
            walls_lds[wave][slot] = mine;
            hits_lds[wave][slot] = SW;                    // none: first 320, one past the last 0
        }
        const int width = live ? max(window1 - window0, 0) : 0;
        int members[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const bool member = width > (k ? 4 << k : 0) && width <= (8 << k);
            const u64 all = __ballot(member);
            if (member) by_width[wave][k][__popcll(all & ((1ULL << slot) - 1))] = (unsigned char)slot;
            members[k] = __popcll(all);
        }
        wave_lds_fence();
        // The linedef at column x, its rays and owned span known: a candidate there if its distance is finite (engine.py:11446-11451).
        // List order is irrelevant: scans break ties on the linedef index.
        auto enter = [&](const SetupWall &q, int x, bool ok, bool g, bool along_high, float d, int owned) {
            const int from = owned & 0xFFFF, to = (owned >> 16) & 0x7FFF;
            const bool p = ok && d > 0 && owned < 0 && x >= from && x < to;
            const bool valid = (q.facts & WF_ONE_SIDED) ? p && (q.facts & WF_FF) : (g || p);
            if (!valid || !finitef(d)) return;
            const int flags = (g ? CF_GEO : 0) | (p ? CF_PROJ : 0) | ((x == from) ? CF_LEDGE : 0) | (along_high ? CF_ALONG_HI : 0) |
                              (((q.facts >> WF_END_SHIFT) == x) ? CF_ENDS_HERE : 0) | (q.facts & WF_SHOWN);
            Cand entry;
            entry.flags = (unsigned short)flags; entry.wall = (unsigned short)q.wall;
            entry.dist = d;
            if ((q.facts & SETUP_MASKED) && p) atomicMin(&masked_hits[x], cand_key(entry));
            const int at = atomicAdd(&counts[x], 1);
            if (at < CAND_MAX) list[(size_t)at * SW + x] = entry;
            // else: the count says so, and the column is listed afresh in the spill pool (note_length, strip_order_kernel)
        };
        auto look = [&](const SetupWall &q, int x, bool &ok, bool &along_high, float &d) -> bool {   // eval_segment's ray test
            const float rx = rays_lds[x].x, ry = rays_lds[x].y;
            const float den = rx * q.segy - ry * q.segx;
            ok = fabsf(den) >= 1e-6f;
            const float safe = ok ? den : 1.0f;
            d = q.numer / safe;
            const float along = (q.offx * ry - q.offy * rx) / safe;
            along_high = along > 0.5f;
            return ok && (d > 0) && (along >= 0) && (along <= 1);
        };
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int lanes_each = 8 << k, groups = 64 / lanes_each;
            const int group = slot / lanes_each, group_lane = slot - group * lanes_each;
            for (int turn = 0; turn < members[k]; turn += groups) {
                const bool taken = turn + group < members[k];
                const int owner = by_width[wave][k][taken ? turn + group : turn];
                const SetupWall q = walls_lds[wave][owner];
                const int x = (q.window & 0xFFFF) + group_lane;
                const bool inside = taken && x < (q.window >> 16);
                bool ok, along_high; float d;
                const bool g = look(q, x, ok, along_high, d) && inside;
                // the nearest blocking linedef each column ray hits, lowest slot on ties, hides billboards
                if (g && q.blocking >= 0) atomicMin(&block_hits[x], ((u64)__float_as_uint(d) << 32) | (u64)(unsigned)q.blocking);
                const unsigned int hits = (unsigned int)(__ballot(g) >> (group * lanes_each)) & (lanes_each == 32 ? ~0u : (1u << lanes_each) - 1u);
                const bool any = hits != 0;
                const int first = any ? x - group_lane + __ffs((int)hits) - 1 : 0, last = any ? x - group_lane + 31 - __clz((int)hits) : SW - 1;
                if (group_lane == 0 && taken && any) hits_lds[wave][owner] = first | ((last + 1) << 16);
                if (inside) enter(q, x, ok, g, along_high, d, setup_owned(q.facts, q.ends, any, first, last));
            }
        }
        for (u64 pending = __ballot(width > 32); pending; pending &= pending - 1) {
            const int owner = __ffsll((long long)pending) - 1;
            const SetupWall q = walls_lds[wave][owner];
            const int from = q.window & 0xFFFF, to = q.window >> 16;
            int first = 0, last = SW - 1; bool any = false;
            for (int x = from + slot; x - slot < to; x += 64) {
                bool ok, along_high; float d;
                const bool g = look(q, x, ok, along_high, d) && x < to;
                if (g && q.blocking >= 0) atomicMin(&block_hits[x], ((u64)__float_as_uint(d) << 32) | (u64)(unsigned)q.blocking);
                const u64 hits = __ballot(g);
                if (slot == 0) wide_hits[wave][(x - from) / 64] = hits;
                if (hits) {
                    if (!any) first = x - slot + __ffsll((long long)hits) - 1;
                    last = x - slot + 63 - __clzll((long long)hits);
                    any = true;
                }
                if (x < to) wide_lds[wave][x] = !(ok && d > 0) ? 0.0f : (along_high ? -d : d);
            }
            if (slot == 0 && any) hits_lds[wave][owner] = first | ((last + 1) << 16);
            const int owned = setup_owned(q.facts, q.ends, any, first, last);
            wave_lds_fence();
            for (int x = from + slot; x < to; x += 64) {
                const float d = wide_lds[wave][x];
                enter(q, x, true, (wide_hits[wave][(x - from) / 64] >> slot) & 1, d < 0.0f, fabsf(d), owned);
            }
            wave_lds_fence();
        }
        wave_lds_fence();
        if (live) {
            const int hits = hits_lds[wave][slot];
            const bool any = (hits >> 16) != 0;
            const int owned = setup_owned(facts, ends, any, any ? hits & 0xFFFF : 0, any ? (hits >> 16) - 1 : SW - 1);
            RecSpan shown;
            shown.pl = (short)(owned & 0xFFFF); shown.pr = (short)((owned >> 16) & 0x7FFF);
            shown.flags = (facts & ~(SETUP_MASKED | SETUP_SPANS)) | (owned < 0 ? WF_HC : 0) | (any ? WF_ANYGEO : 0);
            r.pl = shown.pl; r.pr = shown.pr; r.flags = shown.flags;
            sc.rec[(size_t)local * m->wall_count + w] = r;
            sc.span[(size_t)local * m->wall_count + w] = shown;
        }
        wave_lds_fence();                                // the next share takes the LDS over
    }
    }
    if (!WHOLE) return;
    __syncthreads();
    static_assert(!WHOLE || THREADS >= SW, "wall_setup_kernel: a thread a column");
    if (threadIdx.x < SW) {                              // whole wavefronts
        const int x = threadIdx.x;
        const size_t at = (size_t)local * SW + x;
        sc.block_hit[at] = block_lds[x]; sc.masked_hit[at] = masked_lds[x]; sc.cand_count[at] = count_lds[x];
        note_length(sc, local, x, count_lds[x]);
    }
}

// The candidate list of every column that was given a spill slot, written afresh into the pool: one wavefront per
// column tests the column's ray against every linedef of the map (eval_wall: the same test, on the same per-linedef
// facts, that entered the linedef in wall_setup_kernel) and keeps those with a finite distance, in linedef order.
// Nearly every frame finds no column to do: the work-groups beside the one that orders the strips look.
__device__ __forceinline__ void list_spilled_columns(const DeviceMap &dm, const Scratch &sc, int wavefront, int wavefronts) {
    const gd_map_desc *m = &dm.d;
    const int wanted = *sc.spill_count;
    const int total = wanted < sc.spill_slots ? wanted : sc.spill_slots;
    const int walls = m->wall_count, lane_id = threadIdx.x & 63;
    for (int slot = wavefront; slot < total; slot += wavefronts) {
        const int column = sc.spill_columns[slot];
        const int local = column / SW, x = column - local * SW;
        const LaneCtx &c = sc.ctx[local];
        float rx, ry; ray_direction(c, x, &rx, &ry);
        const RecSpan *spans = sc.span + (size_t)local * walls;
        Cand *list = sc.cand + sc.spill_base + ((size_t)(slot / SW) * SPILL_DEPTH * SW + (size_t)(slot % SW));
        int listed = 0;
        for (int w0 = 0; w0 < walls; w0 += 64) {
            const int w = w0 + lane_id;
            bool keep = false;
            Cand entry;
            if (w < walls) {
                const Eval e = eval_wall(m, c, spans, x, w, rx, ry);
                keep = finitef(e.dist);
                entry.wall = (unsigned short)w;
                entry.flags = (unsigned short)e.flags;
                entry.dist = e.dist;
            }
            const u64 keeps = __ballot(keep);
            const int position = listed + __popcll(keeps & ((1ULL << lane_id) - 1ULL));
            if (keep) {
                if (position < SPILL_DEPTH) list[(size_t)position * SW] = entry;
                else sc.status[STATUS_CAND_OVERFLOW] = 1;
            }
            listed += __popcll(keeps);
        }
        if (lane_id == 0) sc.cand_count[column] = (listed < SPILL_DEPTH ? listed : SPILL_DEPTH) | ((slot + 1) << SPILL_SHIFT);
    }
}

// ---------------------------------------------------------------------------------------------
// flats: engine.py:10956-11171
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ float flat_center(const LaneCtx &c) { return 103.5f + c.pitch_offset; }

// Per pixel: nearest plane among all sectors (engine.py:10981-11024).  Sectors that share a
// plane height share the candidate point, and the distance grows with the plane height, so the
// levels are visited nearest first and the scan stops once a farther level cannot win.
//
// Does the point lie in some sector whose floor (ceiling) is at `level`?  The even-odd test of
// engine.py:10994-11015 over the sectors the point-location grid lists for the point's cell.
__device__ bool flat_level_hit(const DeviceMap &dm, bool is_floor, float level, float px, float py) {
    const gd_map_desc *m = &dm.d;
    int cell;
    const unsigned fine = fine_lookup(m, dm.fine_inverse, px, py, &cell);
    const unsigned kind = FINE_KIND(fine);
    if (kind == FINE_EMPTY) return false;
    if (kind == FINE_DECIDED) return m->sector_heights[2 * (int)(fine & 0xFFFFu) + (is_floor ? 0 : 1)] == level;
    if (cell < 0) cell = grid_cell_of(m, px, py);
    if (cell < 0) return false;
    const int2 range = dm.cell_range[cell];
    for (int it = range.x; it < range.y; ++it) {
        const int4 item = dm.cell_item[it];
        const int s = item.x & ~GRID_ALWAYS_INSIDE;
        if (m->sector_heights[2 * s + (is_floor ? 0 : 1)] != level) continue;
        if ((item.x & GRID_ALWAYS_INSIDE) || inside_edge_copies(dm.cell_edge, item.z, item.w, px, py)) return true;
    }
    return false;
}
//
// The plane levels of one half of the screen (floors or ceilings) as one lane sees them.
struct LevelSide {
    const float *level, *reach, *far;   // plane height, and the bounds of the distance to the sectors of that level
    const float4 *box;                  // the box around them
    const unsigned int *masks;          // the lane's bit sets by bucket (level_bucket), null without
    int count, first, mask_words;       // levels of this half, the first one's bit
    int index_shift, mask_shift;        // where a raster entry keeps the sector's level index and the mask of undecided cells
};
__device__ __forceinline__ LevelSide level_side(const DeviceMap &dm, const Scratch &sc, int local, bool is_floor) {
    const gd_map_desc *m = &dm.d;
    LevelSide side;
    const int total = m->floor_level_count + m->ceil_level_count;
    side.count = is_floor ? m->floor_level_count : m->ceil_level_count;
    side.first = is_floor ? 0 : m->floor_level_count;
    side.level = is_floor ? m->floor_levels : m->ceil_levels;
    side.reach = sc.level_reach + (size_t)local * total + side.first;
    side.far = sc.level_far + (size_t)local * total + side.first;
    side.box = dm.level_box + side.first;
    side.mask_words = level_mask_words(m);
    side.masks = sc.level_masks + (size_t)local * LEVEL_BUCKETS * side.mask_words;
    side.index_shift = is_floor ? 16 : 20;
    side.mask_shift = is_floor ? 0 : FINE_MASK_LEVELS;
    return side;
}

// A hit of a flat probe as one number: distances are positive, so the smallest key is the nearest hit, the lowest sector on ties.
#define PROBE_NONE 0xFFFFFFFFFFFFFFFFULL
__device__ __forceinline__ u64 probe_key(float cd, int sector) { return ((u64)__float_as_uint(cd) << 32) | (unsigned)sector; }
__device__ __forceinline__ float probe_distance(u64 key) { return key == PROBE_NONE ? GD_INF : __uint_as_float((unsigned)(key >> 32)); }
__device__ __forceinline__ int probe_sector(u64 key) { return key == PROBE_NONE ? -1 : (int)(unsigned)key; }

// The sector of plane level k that holds a point, from the coarse grid's cell (-1: located here), -1 if none does: what the
// raster leaves undecided (engine.py:10994-11015).
__device__ __forceinline__ int cell_sector(const DeviceMap &dm, bool is_floor, int k, float level, int cell, float px, float py) {
    const gd_map_desc *m = &dm.d;
    if (cell < 0) cell = grid_cell_of(m, px, py);
    if (cell < 0) return -1;
    const int2 range = dm.cell_range[cell];
    int found = -1;
    for (int it = range.x; it < range.y; ++it) {
        const int4 item = dm.cell_item[it];
        const int s = item.x & ~GRID_ALWAYS_INSIDE;
        const bool same_level = item.y >= 0 ? ((is_floor ? (item.y & 0xFFFF) : (item.y >> 16)) == k)
                                            : (m->sector_heights[2 * s + (is_floor ? 0 : 1)] == level);
        if (!same_level || (found >= 0 && s > found)) continue;
        if ((item.x & GRID_ALWAYS_INSIDE) || inside_edge_copies(dm.cell_edge, item.z, item.w, px, py)) found = s;
    }
    return found;
}

// Does the flat ray of one pixel resolve at all, i.e. does the probe point of some plane level lie in a
// sector of that level (engine.py:10981-11024)?  `plane` is the sector whose plane the wall pass shows at the
// pixel: its own level nearly always answers yes at once.  Where it does not, the levels that the pixel's bucket names are asked, and
// of those only the ones whose probe point meets the box around their sectors are looked up (with all 400 levels of a half looked up,
// one after the other, sprite_pixels_kernel took 0.51 ms for 4096 lanes, now 0.39).
__device__ bool flat_ray_resolves(const DeviceMap &dm, const Scratch &sc, int local, const LaneCtx &c, float rc, float rs, float cc, int y, int plane) {
    const gd_map_desc *m = &dm.d;
    const float delta = (float)y - flat_center(c);
    const bool is_floor = delta > 0;
    const float denom = fmaxf(fabsf(delta), 0.5f);
    const LevelSide side = level_side(dm, sc, local, is_floor);
    const float own = m->sector_heights[2 * plane + (is_floor ? 0 : 1)];
    const unsigned int *row = side.masks + level_bucket((192.0f / denom) / cc) * side.mask_words;
    const int end = side.first + side.count;
    int base = (side.first & ~31) - 32;
    unsigned int bits = 0u;
    for (bool first = true;; first = false) {       // one copy of the test: the own level, then the named ones
        float level = own;
        float4 box = make_float4(-GD_INF, -GD_INF, GD_INF, GD_INF);
        if (!first) {
            while (bits == 0u) {
                base += 32;
                if (base >= end) return false;
                bits = side.mask_words > 0 ? row[base >> 5] : ~0u;
                if (base < side.first) bits &= ~0u << (side.first - base);
                if (base + 32 > end) bits &= (1u << (end - base)) - 1u;
            }
            // the pixels of a wavefront name much the same levels: those that name the first one's next take it together
            const int at = __builtin_amdgcn_readfirstlane(base + __ffs((int)bits) - 1);
            const unsigned int bit = (at & ~31) == base ? 1u << (at & 31) : 0u;
            if (!(bits & bit)) continue;
            bits &= ~bit;
            level = at < m->floor_level_count ? m->floor_levels[at] : m->ceil_levels[at - m->floor_level_count];
            box = dm.level_box[at];
            if (level == own) continue;
        }
        const float height = is_floor ? (c.view_z - level) : (level - c.view_z);
        const float cd = (height * 192.0f / denom) / cc;
        const float px = c.x + rc * cd, py = c.y + rs * cd;
        if (!(height > 0 && finitef(cd) && cd > 0)) continue;
        if (!first && !(px >= box.x && px <= box.z && py >= box.y && py <= box.w)) continue;
        if (flat_level_hit(dm, is_floor, level, px, py)) return true;
    }
}

// One pixel's flat ray, tested by PROBE_LANES lanes of a wavefront (a wavefront takes four pixels, of any lanes): the sector of the
// nearest plane level whose probe point lies in a sector of that level, -1 if there is none (engine.py:10981-11024).  Sectors that
// share a plane height share the probe point.  The lanes list the half's levels that the pixel's bucket names, then
// keep those whose probe point lies in the box around the level's sectors, then look the kept ones up, each step for all of them at
// once: a pixel costs a few rounds of loads, where one thread walking the levels of a map with a level per sector waited
// for some forty, one after the other (98 us a pixel; the flat pass of 512 lanes with 800 plane levels took 1.0 ms, its chain of
// kernels being as long as the slowest pixel of each).
#define PROBE_LANES 16
#define PROBE_GROUPS (64 / PROBE_LANES)
#define PROBE_LEVELS 96     // levels a group can list by their bits; a pixel whose bucket names more tests the bits level by level
#define PROBE_KEPT 32       // kept levels waiting to be looked up: one round and one more
struct ProbeLds {
    unsigned short level[PROBE_GROUPS][PROBE_LEVELS];
    float kept_cd[PROBE_GROUPS][PROBE_KEPT]; unsigned short kept_level[PROBE_GROUPS][PROBE_KEPT];
};
__device__ __forceinline__ int flat_probe_group(const DeviceMap &dm, const Scratch &sc, const gd_lanes_desc &lanes, int local, int n, int x, int y, bool live, ProbeLds *lds) {
    const gd_map_desc *m = &dm.d;
    const LaneCtx &c = sc.ctx[local];
    const int lane_id = threadIdx.x & 63, group = lane_id / PROBE_LANES, slot = lane_id - group * PROBE_LANES;
    const float delta = (float)y - flat_center(c);
    const bool is_floor = delta > 0;
    const float denom = fmaxf(fabsf(delta), 0.5f), cc = dm.cosine_correction[x];
    float rc = lanes.ray_cos[(size_t)n * SW + x], rs = lanes.ray_sin[(size_t)n * SW + x];
    asm volatile("" : "+v"(rc), "+v"(rs));    // waited for here, not in every round behind its branches (flat_select_row)
    const LevelSide side = level_side(dm, sc, local, is_floor);
    const unsigned int *row = side.mask_words > 0 ? side.masks + level_bucket((192.0f / denom) / cc) * side.mask_words : nullptr;
    const u64 group_mask = ((1ULL << PROBE_LANES) - 1) << (group * PROBE_LANES), lower_lanes = (1ULL << lane_id) - 1;
    // the levels the bucket names, listed: each lane takes whole words of the bit set
    int named = live ? side.count : 0;
    bool listed = false;
    if (row) {
        unsigned int bits[2] = {0u, 0u};
        static_assert(LEVEL_MASK_WORDS_MAX <= 2 * PROBE_LANES, "flat_probe_group: two words of a bucket's bit set a lane");
        const int end = side.first + side.count;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int word = slot * 2 + j, base = word * 32;
            if (live && word < side.mask_words) bits[j] = row[word];
            if (base < side.first) bits[j] = base + 32 <= side.first ? 0u : bits[j] & (~0u << (side.first - base));
            if (base + 32 > end) bits[j] = base >= end ? 0u : bits[j] & ((1u << (end - base)) - 1u);
        }
        int at = __popc(bits[0]) + __popc(bits[1]);
        const int own = at;
#pragma unroll
        for (int step = 1; step < PROBE_LANES; step <<= 1) { const int left = __shfl_up(at, step, PROBE_LANES); at += slot >= step ? left : 0; }
        const int total = __shfl(at, PROBE_LANES - 1, PROBE_LANES);
        at -= own;
        listed = total <= PROBE_LEVELS;
        if (listed) {
            named = total;
#pragma unroll
            for (int j = 0; j < 2; ++j)
                for (unsigned int rest = bits[j]; rest; rest &= rest - 1u) lds->level[group][at++] = (unsigned short)(slot * 64 + j * 32 + __ffs((int)rest) - 1 - side.first);
        }
        wave_lds_fence();
    }
    u64 best = PROBE_NONE;
    int kept = 0;
    auto look_up = [&]() {
        wave_lds_fence();
        for (int base = 0; __ballot(base < kept) != 0; base += PROBE_LANES) {
            u64 key = PROBE_NONE;
            if (base + slot < kept) {
                const float cd = lds->kept_cd[group][base + slot];
                const int k = lds->kept_level[group][base + slot];
                const float px = c.x + rc * cd, py = c.y + rs * cd;
                int cell;
                const unsigned fine = fine_lookup(m, dm.fine_inverse, px, py, &cell);
                const unsigned kind = FINE_KIND(fine);
                int s = -1;
                if (kind == FINE_DECIDED) {
                    const int decided = (int)(fine & 0xFFFFu);
                    const unsigned index = (fine >> side.index_shift) & 15u;   // the sector's level index, 15 = not recorded
                    if (index == 15u ? m->sector_heights[2 * decided + (is_floor ? 0 : 1)] == side.level[k] : index == (unsigned)k) s = decided;
                } else if (kind == FINE_UNKNOWN || (kind == FINE_MIXED && ((fine >> (side.mask_shift + k)) & 1u))) {
                    s = cell_sector(dm, is_floor, k, side.level[k], cell, px, py);
                }
                if (s >= 0) key = probe_key(cd, s);
            }
#pragma unroll
            for (int step = 1; step < PROBE_LANES; step <<= 1) {
                const u64 other = ((u64)(unsigned)__shfl_xor((int)(key >> 32), step) << 32) | (unsigned)__shfl_xor((int)(unsigned)key, step);
                key = other < key ? other : key;
            }
            best = key < best ? key : best;
        }
        kept = 0;
        wave_lds_fence();
    };
    for (int base = 0; __ballot(base < named) != 0; base += PROBE_LANES) {
        bool wanted = base + slot < named;
        int k = base + slot;
        if (wanted && listed) k = lds->level[group][base + slot];
        if (wanted && row && !listed) { const int bit = side.first + k; wanted = (row[bit >> 5] >> (bit & 31)) & 1u; }
        float cd = 0.0f;
        if (wanted) {
            const float height = is_floor ? (c.view_z - side.level[k]) : (side.level[k] - c.view_z);
            const float4 box = side.box[k];
            cd = (height * 192.0f / denom) / cc;
            const float px = c.x + rc * cd, py = c.y + rs * cd;
            wanted = height > 0 && finitef(cd) && cd > 0 && px >= box.x && px <= box.z && py >= box.y && py <= box.w && !(cd > probe_distance(best));
        }
        const u64 bits = __ballot(wanted) & group_mask;
        if (wanted) {
            const int at = kept + __popcll(bits & lower_lanes);
            lds->kept_cd[group][at] = cd; lds->kept_level[group][at] = (unsigned short)k;
        }
        kept += __popcll(bits);
        if (__ballot(kept > PROBE_KEPT - PROBE_LANES) != 0) look_up();
    }
    look_up();
    return probe_sector(best);
}

// 64 neighbouring pixels of ONE row of one lane's screen, a wavefront's lane each (wanted or not: every lane takes part);
// the sector of each as in flat_probe_group.  The 64 rays share the row, so a level's perpendicular distance is worked out once
// (by the lane whose turn it is), and the levels none of the 64 can reach are never listed: those whose sectors lie nearer or
// farther than any of their probe points, or beside the wedge the 64 rays span (with a level per sector that leaves a few of
// forty).  The listed ones are looked up in the raster one after the other, ROW_BATCH loads in flight; what the raster leaves
// undecided (a point near a linedef) waits in a queue in LDS and is settled at the end by all lanes together, unless a nearer
// level has been found by then.  (Settled where it came up, a single undecided pixel held up its whole wavefront for
// the three dependent loads of the coarse grid, at nearly every level.)
#define ROW_LIST 96         // levels listed at a time: 32 and one more round of 64
#define ROW_BATCH 4         // levels looked up together
#define ROW_QUEUE (64 + 64 * ROW_BATCH)   // undecided probes waiting: at most 64 before a batch of levels
#define ROW_NAMED 256       // levels listed by their bits; where the buckets name more, the bits are tested level by level
struct RowLds {
    float4 level[ROW_LIST];                                    // perpendicular distance, least distance to a sector, greatest, bits(index)
    float queue_cd[ROW_QUEUE]; unsigned queue_who[ROW_QUEUE];   // lane << 16 | level index
    unsigned short named[ROW_NAMED];
    u64 best[64];
};
// MASKS: the map has enough plane levels for the per-bucket bit sets (level_mask_words() > 0).
template <bool MASKS>
__device__ __forceinline__ int flat_select_row(const DeviceMap &dm, const Scratch &sc, const gd_lanes_desc &lanes, int local, int n, int x, int y, bool wanted, RowLds *lds) {
    const gd_map_desc *m = &dm.d;
    const LaneCtx &c = sc.ctx[local];
    const int lane_id = threadIdx.x & 63;
    const u64 lower_lanes = (1ULL << lane_id) - 1;
    const float delta = (float)y - flat_center(c);
    const bool is_floor = __builtin_amdgcn_readfirstlane((int)(delta > 0)) != 0;   // the same in every lane, like the row
    const float denom = fmaxf(fabsf(delta), 0.5f);
    float cc = dm.cosine_correction[x];
    float rc = lanes.ray_cos[(size_t)n * SW + x], rs = lanes.ray_sin[(size_t)n * SW + x];
    const LevelSide side = level_side(dm, sc, local, is_floor);
    // cd = perpendicular / cc below is the hot division.  With y = RN(1 / cc), q = RN(p * y) is within
    // one ulp of p / cc, and RN(q + RN(p - cc * q) * y) is then the correctly rounded quotient
    // (Markstein's theorem; the inner product is exact in an FMA) as long as nothing over- or
    // underflows, which the range tests on both operands ensure.
    float inv_cc = dm.inverse_cosine[x];
    // Waited for here.  Where a probe first asks for one of them behind a branch, the compiler waits for all loads at every probe, the raster
    // loads of the probes before among them, which then come one by one and not ROW_BATCH together.
    asm volatile("" : "+v"(cc), "+v"(rc), "+v"(rs), "+v"(inv_cc));
    const bool cc_plain = cc >= 0.5f && cc <= 1.0f;
    const float inv_fine = dm.fine_inverse;       // a reciprocal is fine here: see fine_lookup_cells
    // the probe point camera + ray * cd in raster cell units, as one multiply-add per axis
    const float cell_x0 = (c.x - m->grid_min_x) * inv_fine, cell_y0 = (c.y - m->grid_min_y) * inv_fine;
    const float cell_dx = rc * inv_fine, cell_dy = rs * inv_fine;
    // perpendicular / (smallest cc of the 64) bounds every cd from above, perpendicular / (largest cc) from below
    const float reach_scale = dm.strip_reach_scale[__builtin_amdgcn_readfirstlane(x >> 6)];
    const float far_scale = dm.strip_far_scale[__builtin_amdgcn_readfirstlane(x >> 6)];
    // the wedge's leftmost and rightmost ray; rays turn clockwise from left to right
    const float left_c = bcast(rc, 0), left_s = bcast(rs, 0), right_c = bcast(rc, 63), right_s = bcast(rs, 63);
    u64 best = PROBE_NONE;
    bool done = !wanted;
    int listed = 0, queued = 0;                   // the same in every lane
    auto settle_queue = [&]() {
        if (queued == 0) return;
        lds->best[lane_id] = best;
        wave_lds_fence();
        for (int base = 0; base < queued; base += 64) {
            const int e = base + lane_id;
            const bool live = e < queued;
            const unsigned who = live ? lds->queue_who[e] : 0u;
            const int owner = (int)(who >> 16), k = (int)(who & 0xFFFFu);
            const float cd = live ? lds->queue_cd[e] : 0.0f;
            const float o_rc = __shfl(rc, owner), o_rs = __shfl(rs, owner);
            if (live && !(cd > probe_distance(lds->best[owner]))) {
                const int s = cell_sector(dm, is_floor, k, side.level[k], -1, c.x + o_rc * cd, c.y + o_rs * cd);
                if (s >= 0) atomicMin(&lds->best[owner], probe_key(cd, s));
            }
        }
        wave_lds_fence();
        best = lds->best[lane_id];
        queued = 0;
    };
    auto probe_listed = [&]() {
        wave_lds_fence();
        for (int j0 = 0; j0 < listed; j0 += ROW_BATCH) {
            if (__ballot(!done) == 0) break;
            if (queued > 64) settle_queue();
            float cdv[ROW_BATCH]; unsigned finev[ROW_BATCH]; int kv[ROW_BATCH];
#pragma unroll
            for (int j = 0; j < ROW_BATCH; ++j) {
                cdv[j] = -1.0f; finev[j] = 0x40000000u; kv[j] = 0;                    // empty: nothing there
                if (j0 + j >= listed) continue;                                       // the same in every lane
                const float4 entry = lds->level[j0 + j];
                kv[j] = __float_as_int(entry.w);
                const float perpendicular = entry.x;
                float cd;
                if (cc_plain && perpendicular >= 1e-18f && perpendicular <= 1e18f) {
                    const float q = perpendicular * inv_cc;
                    cd = __builtin_fmaf(__builtin_fmaf(-cc, q, perpendicular), inv_cc, q);
                } else {
                    cd = perpendicular / cc;
                }
                cdv[j] = cd;
                if (cd > probe_distance(best)) done = true;      // later levels are at least this far
                if (done || !(finitef(cd) && cd > 0) || cd < entry.y || cd > entry.z) continue;
                int cell;
                finev[j] = fine_lookup_cells(m, __builtin_fmaf(cd, cell_dx, cell_x0), __builtin_fmaf(cd, cell_dy, cell_y0), &cell);
            }
#pragma unroll
            for (int j = 0; j < ROW_BATCH; ++j) {
                const unsigned fine = finev[j], kind = FINE_KIND(fine);
                const int k = kv[j];
                bool undecided = false;
                if (kind == FINE_DECIDED) {
                    const int s = (int)(fine & 0xFFFFu);
                    const unsigned index = (fine >> side.index_shift) & 15u;   // the sector's level index, 15 = not recorded
                    if (index == 15u ? m->sector_heights[2 * s + (is_floor ? 0 : 1)] == side.level[k] : index == (unsigned)k) {
                        const u64 key = probe_key(cdv[j], s);
                        best = key < best ? key : best;
                    }
                } else if (kind == FINE_UNKNOWN || (kind == FINE_MIXED && ((fine >> (side.mask_shift + k)) & 1u))) {
                    undecided = true;
                }
                const u64 waiting = __ballot(undecided);
                if (undecided) {
                    const int at = queued + __popcll(waiting & lower_lanes);
                    lds->queue_cd[at] = cdv[j]; lds->queue_who[at] = ((unsigned)lane_id << 16) | (unsigned)k;
                }
                queued += __popcll(waiting);
            }
        }
        listed = 0;
        wave_lds_fence();
    };
    // The levels the buckets of the 64 scales name: lane j joins word j of their bit sets.
    int named = side.count;
    bool by_bits = false;
    unsigned int joined_word = 0u;
    if (MASKS) {
        const int bucket = level_bucket((192.0f / denom) / cc);
        int lowest = bucket, highest = bucket;
#pragma unroll
        for (int step = 1; step < 64; step <<= 1) { lowest = min(lowest, __shfl_xor(lowest, step)); highest = max(highest, __shfl_xor(highest, step)); }
        if (lane_id < side.mask_words) for (int b = lowest; b <= highest; ++b) joined_word |= side.masks[b * side.mask_words + lane_id];
        unsigned int bits = joined_word;
        const int base = lane_id * 32, end = side.first + side.count;
        if (base < side.first) bits = base + 32 <= side.first ? 0u : bits & (~0u << (side.first - base));
        if (base + 32 > end) bits = base >= end ? 0u : bits & ((1u << (end - base)) - 1u);
        int at = __popc(bits);
        const int own = at;
#pragma unroll
        for (int step = 1; step < LEVEL_MASK_WORDS_MAX; step <<= 1) { const int left = __shfl_up(at, step); at += lane_id >= step ? left : 0; }
        const int total = bcast(at, LEVEL_MASK_WORDS_MAX - 1);
        at -= own;
        by_bits = total <= ROW_NAMED;
        if (by_bits) {
            named = total;
            for (; bits; bits &= bits - 1u) lds->named[at++] = (unsigned short)(base + __ffs((int)bits) - 1 - side.first);
        }
        wave_lds_fence();
    }
    for (int base = 0; base < named; base += 64) {
        if (__ballot(!done) == 0) break;
        bool reachable = base + lane_id < named;
        int k = base + lane_id;
        if (MASKS) {
            if (by_bits) { if (reachable) k = lds->named[base + lane_id]; }
            else {
                const int bit = side.first + k;
                const unsigned int word = (unsigned)__shfl((int)joined_word, (bit >> 5) & 63);   // lanes past the last word hold zeros
                reachable = reachable && ((word >> (bit & 31)) & 1u);
            }
        }
        float4 entry = make_float4(0.0f, 0.0f, 0.0f, __int_as_float(k));
        if (reachable) {
            const float height = is_floor ? (c.view_z - side.level[k]) : (side.level[k] - c.view_z);
            const float4 box = side.box[k];
            entry.x = height * 192.0f / denom; entry.y = side.reach[k]; entry.z = side.far[k];
            // the box's corner farthest to the right of the leftmost ray, farthest to the left of the rightmost one, and farthest ahead
            // (a map unit to spare: the rays are unit vectors, the coordinates below 2^15)
            const float x0 = box.x - c.x, x1 = box.z - c.x, y0 = box.y - c.y, y1 = box.w - c.y;
            const float beyond_left = fminf(left_c * y0, left_c * y1) - fmaxf(left_s * x0, left_s * x1);
            const float beyond_right = fmaxf(right_c * y0, right_c * y1) - fminf(right_s * x0, right_s * x1);
            reachable = height > 0 && entry.x > 0 && !(entry.x * reach_scale < entry.y) && !(entry.x * far_scale > entry.z) &&
                        !(beyond_left > 1.0f) && !(beyond_right < -1.0f);
        }
        const u64 bits = __ballot(reachable);
        if (reachable) lds->level[listed + __popcll(bits & lower_lanes)] = entry;
        listed += __popcll(bits);
        if (listed > ROW_LIST - 64) probe_listed();
    }
    probe_listed();
    settle_queue();
    return probe_sector(best);
}

// The flat pass runs after the walls and only where its result can matter.  A pixel a wall tier filled never
// shows it; a pixel a plane of the wall pass claimed only asks whether the flat ray resolved at all, and only
// where a sprite stands behind the plane with no sprite clip recorded, which the sprite pass finds out for
// itself (flat_ray_resolves); the few pixels left (columns whose traversal left a gap) show the flat pass's
// picture.  wall_raster_kernel lists their columns, of all lanes together: most lanes have none, some have hundreds.
// flat_gap_kernel, a work-group per half of the screen of a listed column, selects them.
//
// Then, column by column, the vertical repair (engine.py:11026-11083).  An unresolved
// pixel takes the sector of the next resolved pixel below it in its half of the screen; when that sector is not the camera's,
// the pixel is its own left and right anchor in the horizontal repair (engine.py:11085-11135), which then leaves
// it as it is: such a pixel is settled here and its row needs no further work.  Only the rows of the others (no
// resolved pixel below, or the camera's own sector) are noted for the row kernels (flat_span_select_kernel,
// flat_tail_kernel, flat_span_finish_kernel).

// A lane's half of the screen gets rows to repair: it joins the work list of the row kernels when it gets its first.
__device__ __forceinline__ void note_row(const Scratch &sc, int local, int half, int y) {
    int *span = sc.flat_span + (size_t)local * 4 + 2 * half;
    atomicMax(&span[1], y);
    if (atomicMin(&span[0], y) == VH) sc.flat_spans[atomicAdd(sc.flat_span_count, 1)] = (local << 1) | half;
}

// GAP_WAVES wavefronts a column's half of the screen, which probe four rows each at a time, from the topmost gap pixel down, until the lowest one is
// past and, if any is unresolved, a resolved pixel below the last of those is found (or the half ends).  The kernel lasts as long as
// its slowest halves, rounds of probes one after the other.  Rows between gap pixels, and below them as far as the last round
// reaches, are probed along with them, needed or not: 93 % of the halves hold an unresolved pixel, and the round lasts as long either way.
// (Gap pixels first, then the rows between and below, the halves of a column one after the other: 42 us where this takes 24 at 256 lanes of 800
// linedefs, 83 and 65 at 512 lanes of 4000.)
template <int GAP_WAVES>
__global__ void __launch_bounds__(64 * GAP_WAVES) flat_gap_kernel(DeviceMap dm, gd_lanes_desc lanes, int lane_base, Scratch sc) {
    __shared__ ProbeLds probe_lds[GAP_WAVES];
    __shared__ short row_sector[VH];                  // the sector of each row's pixel, -1 unresolved
    __shared__ int unresolved_first, unresolved_last, resolved_last;
    const int total = *sc.gap_column_count;
    const int wave = threadIdx.x >> 6, lane_id = threadIdx.x & 63, group = wave * PROBE_GROUPS + lane_id / PROBE_LANES;
    const bool speaks = (lane_id & (PROBE_LANES - 1)) == 0;
    constexpr int ROWS = GAP_WAVES * PROBE_GROUPS;
    for (int task = blockIdx.x; task < 2 * total; task += gridDim.x) {
        const int2 packed = sc.gap_columns[task >> 1];
        const int half = task & 1, x = packed.x & 511, local = packed.x >> 9;
        const LaneCtx &c = sc.ctx[local];
        const int n = lane_base + local, last_ceiling_row = c.last_ceiling_row;
        const int half_end = half ? VH - 1 : last_ceiling_row;
        const int lo = max(packed.y & 255, half ? last_ceiling_row + 1 : 0), hi = min((packed.y >> 8) - 1, half_end);
        if (lo > hi) continue;                        // the same in the whole block, like everything that steers it here
        const unsigned int *meta = sc.meta + (size_t)local * VH * SW + x;
        unsigned short *sector = sc.flat_sector + (size_t)local * VH * SW + x;
        unsigned char *flags = sc.flat_flags + (size_t)local * VH * SW + x;
        __syncthreads();                              // nobody reads the previous half's rows any more
        if (threadIdx.x == 0) { unresolved_first = VH; unresolved_last = -1; resolved_last = -1; }
        int rows_end = lo;
        for (bool more = true; more && rows_end <= half_end;) {
            __syncthreads();                          // the bounds are set, and everyone has seen the last round's
            const int y = rows_end + group;
            const bool live = y <= half_end, shown = y <= hi && gap_pixel(meta[(size_t)y * SW]);
            const int s = flat_probe_group(dm, sc, lanes, local, n, x, live ? y : lo, live, &probe_lds[wave]);
            if (live && speaks) {
                row_sector[y] = (short)s;
                if (s >= 0) atomicMax(&resolved_last, y);
                if (shown) {
                    sector[(size_t)y * SW] = (unsigned short)(s < 0 ? c.sector : s);
                    flags[(size_t)y * SW] = s < 0 ? 1 : 0;
                    if (s < 0) { atomicMin(&unresolved_first, y); atomicMax(&unresolved_last, y); }
                }
            }
            rows_end += ROWS;
            __syncthreads();
            more = rows_end <= hi || (unresolved_last >= 0 && resolved_last < unresolved_last);
        }
        rows_end = min(rows_end, half_end + 1);
        for (int y = unresolved_first + (int)threadIdx.x; y <= unresolved_last; y += blockDim.x) {
            if (row_sector[y] != -1 || !gap_pixel(meta[(size_t)y * SW])) continue;
            int below = -1;
            for (int j = y + 1; j < rows_end && below < 0; ++j) below = row_sector[j];
            if (below >= 0 && below != c.sector) {
                sector[(size_t)y * SW] = (unsigned short)below;
                flags[(size_t)y * SW] = (unsigned char)(1 | 2 | 4 | 8);
            } else {
                note_row(sc, local, half, y);
            }
        }
    }
}

// The lanes' row ranges are final once every listed column is repaired: their rows join the work list that
// flat_span_select_kernel deals out evenly, whichever lanes they come from, and those below them flat_tail_kernel's.  One wavefront per lane; a
// work-group takes room in the lists for all of its lanes at once (each for itself: 18 us where half of 2048 lanes have rows, now 12; by sixteen lanes a
// work-group 6, but at 4096 lanes such a one waits 0.2 ms for room beside the shading).
#define ROWS_LANES 4
__global__ void __launch_bounds__(64 * ROWS_LANES) flat_rows_kernel(int lane_count, Scratch sc) {
    __shared__ int wanted[2][ROWS_LANES], base[2];
    const int wave = threadIdx.x >> 6, lane_id = threadIdx.x & 63, local = blockIdx.x * ROWS_LANES + wave;
    int lo0 = VH, hi0 = -1, lo1 = VH, hi1 = -1, last_ceiling_row = 0;
    if (local < lane_count) {
        const int4 span = *reinterpret_cast<const int4 *>(sc.flat_span + (size_t)local * 4);
        lo0 = span.x; hi0 = span.y; lo1 = span.z; hi1 = span.w;
        last_ceiling_row = sc.ctx[local].last_ceiling_row;
    }
    const int rows0 = hi0 < lo0 ? 0 : hi0 - lo0 + 1, rows1 = hi1 < lo1 ? 0 : hi1 - lo1 + 1;
    const int below0 = rows0 == 0 ? 0 : last_ceiling_row - hi0, below1 = rows1 == 0 ? 0 : VH - 1 - hi1;
    if (lane_id == 0) { wanted[0][wave] = rows0 + rows1; wanted[1][wave] = below0 + below1; }
    __syncthreads();
    if (threadIdx.x < 2) {
        int total = 0;
        for (int k = 0; k < ROWS_LANES; ++k) { const int own = wanted[threadIdx.x][k]; wanted[threadIdx.x][k] = total; total += own; }
        base[threadIdx.x] = total ? atomicAdd(&sc.flat_row_count[threadIdx.x], total) : 0;
    }
    __syncthreads();
    if (rows0 + rows1 == 0) return;                  // the same in the whole wavefront
    int *rows = sc.flat_rows + base[0] + wanted[0][wave], *below = sc.flat_rows + (size_t)lane_count * VH - 1 - (base[1] + wanted[1][wave]);
    for (int r = lane_id; r < rows0 + rows1; r += 64) rows[r] = (local << 8) | (r < rows0 ? lo0 + r : lo1 + (r - rows0));
    for (int r = lane_id; r < below0 + below1; r += 64) below[-r] = (local << 8) | (r < below0 ? hi0 + 1 + r : hi1 + 1 + (r - below0));
    for (int x = lane_id; x < 2 * SW; x += 64)
        if (x < SW ? rows0 > 0 : rows1 > 0) sc.flat_tail[(size_t)local * 2 * SW + x] = ~0u;
}

// Small per-sector / per-texture tables staged in LDS by the kernels whose inner loops chase
// them (a dependent global gather costs ~500 cycles, an LDS read ~60).  Sectors or textures
// beyond the staged count fall back to the global arrays.
struct Tables {
    const gd_map_desc *m;
    const float4 *sector;          // floor, ceiling, light, bits(floor_tex | ceil_tex << 16)
    const unsigned char *tex_bits; // floor(log2 width) | floor(log2 height) << 4
    const unsigned int *tex_odd;   // bit t: the width of texture t is no power of two
    int sector_cached, tex_cached;
    bool all_cached = false;       // a kernel's constant: every sector and texture of the map is staged
    __device__ __forceinline__ float floor_h(int s) const { return all_cached || s < sector_cached ? sector[s].x : m->sector_heights[2 * s]; }
    __device__ __forceinline__ float ceil_h(int s) const { return all_cached || s < sector_cached ? sector[s].y : m->sector_heights[2 * s + 1]; }
    __device__ __forceinline__ float light(int s) const { return all_cached || s < sector_cached ? sector[s].z : m->sector_lights[s]; }
    __device__ __forceinline__ int floor_tex(int s) const { return all_cached || s < sector_cached ? (int)(__float_as_uint(sector[s].w) & 0xFFFFu) : m->sector_floor_tex[s]; }
    __device__ __forceinline__ int ceil_tex(int s) const { return all_cached || s < sector_cached ? (int)(__float_as_uint(sector[s].w) >> 16) : m->sector_ceil_tex[s]; }
    __device__ __forceinline__ int width_bits(int t) const { return all_cached || t < tex_cached ? (tex_bits[t] & 15) : ilog2(m->tex_w[t]); }
    __device__ __forceinline__ int height_bits(int t) const { return all_cached || t < tex_cached ? (tex_bits[t] >> 4) : ilog2(m->tex_h[t]); }
    // Texture column of a wall: torch.remainder(u, width) (engine.py:12792-12798).  Widths are powers of two
    // on most maps, where the remainder is a mask; WAD textures of other widths take the division.
    __device__ __forceinline__ i64 wrap_column(int t, i64 u) const {
        const bool odd = all_cached || t < tex_cached ? ((tex_odd[t >> 5] >> (t & 31)) & 1u) != 0 : (m->tex_w[t] & (m->tex_w[t] - 1)) != 0;
        if (!odd) return u & (i64)((1 << width_bits(t)) - 1);
        const i64 width = m->tex_w[t];
        const i64 r = u - tdiv(u, width) * width;
        return r < 0 ? r + width : r;
    }
};

// Cooperative fill of the LDS tables by the whole block (call before a __syncthreads()).
struct TexLds { unsigned char bits[LDS_TEXTURES]; unsigned int odd[LDS_TEXTURES / 32]; };
__device__ __forceinline__ void stage_tables(const gd_map_desc *m, float4 *sector_lds, TexLds *tex_lds, Tables &tb) {
    int sectors = m->sector_count < LDS_SECTORS ? m->sector_count : LDS_SECTORS;
    int textures = m->texture_count < LDS_TEXTURES ? m->texture_count : LDS_TEXTURES;
#pragma unroll 4
    for (int s = threadIdx.x; s < sectors; s += blockDim.x) {
        float4 v;
        v.x = m->sector_heights[2 * s]; v.y = m->sector_heights[2 * s + 1]; v.z = m->sector_lights[s];
        v.w = __uint_as_float(((unsigned)m->sector_floor_tex[s] & 0xFFFFu) | ((unsigned)m->sector_ceil_tex[s] << 16));
        sector_lds[s] = v;
    }
    // Whole wavefronts, a texture a lane.  With a thread that went over a word's textures by itself every work-group of wall_raster_kernel began with 32 loads one
    // after the other (and the colormap four bytes at a time); wall_geometry_kernel and it together, then / now: 16 lanes on the 2000-linedef map 80 / 75 us, 256
    // 139 / 130, 2048 lanes on the 320-linedef map 354 / 291, 4096 on the 4000-linedef map 1208 / 1140.
    for (int first = threadIdx.x & ~63; first < LDS_TEXTURES; first += blockDim.x) {
        const int lane = threadIdx.x & 63, t = first + lane;
        const bool there = t < textures;
        const int width = there ? m->tex_w[t] : 1, height = there ? m->tex_h[t] : 1;
        if (there) tex_lds->bits[t] = (unsigned char)(ilog2(width) | (ilog2(height) << 4));
        const u64 odd = __ballot((width & (width - 1)) != 0);
        if (lane < 2 && first / 32 + lane < LDS_TEXTURES / 32) tex_lds->odd[first / 32 + lane] = (unsigned int)(odd >> (32 * lane));
    }
    tb.m = m; tb.sector = sector_lds; tb.tex_bits = tex_lds->bits; tb.tex_odd = tex_lds->odd; tb.sector_cached = sectors; tb.tex_cached = textures;
}

// engine.py:10879-10954
__device__ __forceinline__ void flat_texture_coordinates(const Tables &tb, const LaneCtx &c, int texture_id, float plane_height, int px, int py, i64 *u, i64 *v) {
    int width_bits = tb.width_bits(texture_id);
    int height_bits = tb.height_bits(texture_id);
    i64 xscale = shl64(1, 32 - width_bits), yscale = shl64(1, 32 - height_bits);
    i64 xstep_scale = tdiv(mul64(xscale, c.vsin), FOCAL_X_FIXED);
    i64 ystep_scale = tdiv(mul64(yscale, c.vcos), FOCAL_X_FIXED);
    i64 flat_column = (i64)px - (SW / 2 - 1);
    i64 basexfrac = (mul64(xscale, c.vcos) >> 16) + mul64(flat_column, xstep_scale);
    i64 baseyfrac = (mul64(yscale, -c.vsin) >> 16) + mul64(flat_column, ystep_scale);
    i64 pviewx = mul64(xscale, c.view_x_fixed) >> 16;
    i64 pviewy = mul64(yscale, -c.view_y_fixed) >> 16;
    i64 center_row = c.center_fixed >> 16;
    i64 pixel_y_fixed = (i64)py * FIXED_UNIT;
    i64 den = (py < center_row) ? (c.center_fixed - pixel_y_fixed - FIXED_UNIT / 2) : (pixel_y_fixed - c.center_fixed + FIXED_UNIT / 2);
    den = max64(den, 1);
    bool overflow = den <= (FOCAL_Y_FIXED >> 15);
    i64 yslope = tdiv(FOCAL_Y_FIXED << 16, den);
    if (overflow) yslope = (1LL << 31) - 1;
    i64 plane_height_fixed = round_to_i64(plane_height * 65536.0f);
    i64 distance = mul64(plane_height_fixed, yslope) >> 16;
    i64 xfrac = ((mul64(distance, basexfrac) >> 16) + pviewx) & UINT32_MASK;
    i64 yfrac = ((mul64(distance, baseyfrac) >> 16) + pviewy) & UINT32_MASK;
    *u = xfrac >> (32 - width_bits);
    *v = yfrac >> (32 - height_bits);
}

// engine.py:10588-10616
__device__ __forceinline__ unsigned char plane_colormap(const unsigned char *colormap, const LaneCtx &c, unsigned char index, float light, float plane_height, int py) {
    i64 plane_height_fixed = round_to_i64(plane_height * 65536.0f);
    i64 glob = min64(tdiv(FLOOR_VISIBILITY_FIXED << 16, max64(plane_height_fixed, 1)), (1LL << 31) - 1);
    i64 row = c.center_fixed - (i64)py * FIXED_UNIT;
    if (row < 0) row = -row;
    i64 visibility = min64(mul64(glob, row) >> 16, 24 * FIXED_UNIT);
    i64 plane_shade = 64 * FIXED_UNIT - ((i64)light + 12) * (FIXED_UNIT / 4);
    i64 shade = clampi((plane_shade - visibility) >> 16, 0, 31);
    return colormap[shade * 256 + index];
}

__device__ __forceinline__ unsigned char flat_pixel(const Tables &tb, const unsigned char *colormap, const LaneCtx &c, int sector, bool is_floor, int px, int py) {
    const gd_map_desc *m = tb.m;
    float plane_height = is_floor ? (c.view_z - tb.floor_h(sector)) : (tb.ceil_h(sector) - c.view_z);
    int texture = is_floor ? tb.floor_tex(sector) : tb.ceil_tex(sector);
    i64 u, v;
    flat_texture_coordinates(tb, c, texture, plane_height, px, py, &u, &v);
    unsigned char index = m->tex_atlas[((size_t)texture * m->tex_max_h + v) * m->tex_max_w + u];
    float light = tb.light(sector) + (float)(c.flash_light * 16);
    return plane_colormap(colormap, c, index, light, plane_height, py);
}

// flat_pixel with every division looked up: the lane's per-level, per-row and per-size tables
// hold exactly the quotients flat_texture_coordinates and plane_colormap would compute, and a
// product with a power-of-two texture scale is a shift.
struct LaneTables {
    const i64 *level_plane;   // this lane's [levels][2]
    const i64 *step_scale;    // this lane's [3][2][16]
    int floors;
};
// Returns the texel's offset in the texture atlas and the colormap row, so that a caller can
// have several texel loads in flight before it needs any of them.
__device__ __forceinline__ size_t flat_sample_tabled(const Tables &tb, const LaneCtx &c, const LaneTables &lt,
                                                     i64 yslope, int level_index, int sector, bool is_floor, int px, int py, int *colormap_row) {
    const gd_map_desc *m = tb.m;
    const int texture = is_floor ? tb.floor_tex(sector) : tb.ceil_tex(sector);
    const int width_bits = tb.width_bits(texture), height_bits = tb.height_bits(texture);
    const i64 *plane = lt.level_plane + 2 * (is_floor ? level_index : lt.floors + level_index);
    const i64 plane_height_fixed = plane[0], glob = plane[1];
    // The same integers as flat_texture_coordinates, with narrower multiplies: base + (px - 159) * step is
    // (base - 159 * step) + px * step; the row slope and the visibility factor are below 2^31 and not negative
    // (lane_tables_kernel clamps both); of distance * basefrac only bits 16..47 reach the texel coordinate.
    const i64 xstep_scale = lt.step_scale[width_bits], ystep_scale = lt.step_scale[16 + height_bits];
    const i64 basexfrac = lt.step_scale[32 + width_bits] + mul64_u32(xstep_scale, (unsigned)px);
    const i64 baseyfrac = lt.step_scale[48 + height_bits] + mul64_u32(ystep_scale, (unsigned)px);
    const unsigned pviewx = (unsigned)lt.step_scale[64 + width_bits], pviewy = (unsigned)lt.step_scale[80 + height_bits];
    const i64 distance = mul64_u32(plane_height_fixed, (unsigned)yslope) >> 16;
    const unsigned xfrac = mul64_bits_16_47(distance, basexfrac) + pviewx;
    const unsigned yfrac = mul64_bits_16_47(distance, baseyfrac) + pviewy;
    const unsigned u = (xfrac >> (31 - width_bits)) >> 1, v = (yfrac >> (31 - height_bits)) >> 1;   // two shifts: a size of one shifts by 32
    const float light = tb.light(sector) + (float)(c.flash_light * 16);
    i64 row = c.center_fixed - (i64)py * FIXED_UNIT;
    if (row < 0) row = -row;
    const i64 visibility = min64(mul64_u32(row, (unsigned)glob) >> 16, 24 * FIXED_UNIT);
    const i64 plane_shade = 64 * FIXED_UNIT - ((i64)light + 12) * (FIXED_UNIT / 4);
    *colormap_row = (int)clampi((plane_shade - visibility) >> 16, 0, 31);
    return (size_t)(((unsigned)texture * (unsigned)m->tex_max_h + v) * (unsigned)m->tex_max_w + u);   // the atlas is below 4 GiB (checked at create)
}

// flat_sample_tabled for neighbouring pixels of one row that show the same plane.  Of distance * (base + x * step) only bits 16..47 are
// looked at, and distance * base + x * (distance * step) is the same number modulo 2^48: both products are worked out once
// for the run, and a pixel costs two 24-bit multiply-adds an axis.
// a * b + c of 24-bit factors, whatever lies above their 24 bits.  Written out: where only the sum's lower 24 bits are used the compiler
// takes a 32-bit multiplication, which runs at a quarter of the rate.
__device__ __forceinline__ unsigned mad24(unsigned a, unsigned b, unsigned c) {
    unsigned sum;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(sum) : "v"(a), "v"(b), "v"(c));
    return sum;
}
struct PlaneSpan {
    uint4 start;         // the fraction at the strip's first column, its lower and upper 24 bits: horizontal, then vertical
    uint4 step;          // what a column adds, likewise; the four upper bytes: 24 - log2 width, colormap row, 24 - log2 height, nothing
    unsigned texture;    // the texture's first texel in the atlas (which is below 4 GiB: checked at create)
    // the texel `column` (0..63) columns into the strip
    __device__ __forceinline__ unsigned texel(unsigned column, unsigned atlas_width) const {
        const unsigned x = mad24(step.y, column, start.y) + (mad24(step.x, column, start.x) >> 24);
        const unsigned y = mad24(step.w, column, start.w) + (mad24(step.z, column, start.z) >> 24);
        return texture + __umul24((y & 0xFFFFFFu) >> (step.z >> 24), atlas_width) + ((x & 0xFFFFFFu) >> (step.x >> 24));
    }
    __device__ __forceinline__ unsigned colormap_row() const { return step.y >> 24; }
};
__device__ __forceinline__ PlaneSpan plane_span(const DeviceMap &dm, const Scratch &sc, const LaneCtx &c, int local, int sector, bool is_floor, int x_first, int y) {
    const gd_map_desc *m = &dm.d;
    const int texture = is_floor ? m->sector_floor_tex[sector] : m->sector_ceil_tex[sector];
    const float light = m->sector_lights[sector] + (float)(c.flash_light * 16);
    const i64 yslope = sc.row_slope[(size_t)local * VH + y];
    i64 plane_height_fixed, glob;
    if (dm.sector_level) {       // the lane's table of plane levels
        const int floors = m->floor_level_count, levels = floors + m->ceil_level_count;
        const unsigned int pair = dm.sector_level[sector];
        const longlong2 plane = reinterpret_cast<const longlong2 *>(sc.level_plane)[(size_t)local * levels + (is_floor ? (int)(pair & 0xFFFFu) : floors + (int)(pair >> 16))];
        plane_height_fixed = plane.x; glob = plane.y;
    } else {
        plane_height_fixed = round_to_i64((is_floor ? c.view_z - m->sector_heights[2 * sector] : m->sector_heights[2 * sector + 1] - c.view_z) * 65536.0f);
        glob = min64(tdiv(FLOOR_VISIBILITY_FIXED << 16, max64(plane_height_fixed, 1)), (1LL << 31) - 1);
    }
    const int width_bits = ilog2(m->tex_w[texture]), height_bits = ilog2(m->tex_h[texture]);
    const i64 *scale = sc.step_scale + (size_t)local * STEP_TABLE;
    const i64 xstep = scale[width_bits], ystep = scale[16 + height_bits];
    // the same integers as flat_texture_coordinates: base + (x - 159) * step is (base - 159 * step) + x * step; the row slope and the
    // visibility factor are below 2^31 and not negative (lane_tables_kernel clamps both)
    const u64 distance = (u64)(mul64_u32(plane_height_fixed, (unsigned)yslope) >> 16);
    const u64 xadd = distance * (u64)xstep, yadd = distance * (u64)ystep;
    // the camera's offset in the texture is added to bits 16..47
    const u64 x = distance * (u64)(scale[32 + width_bits] + mul64_u32(xstep, (unsigned)x_first)) + ((u64)scale[64 + width_bits] << 16);
    const u64 v = distance * (u64)(scale[48 + height_bits] + mul64_u32(ystep, (unsigned)x_first)) + ((u64)scale[80 + height_bits] << 16);
    i64 row = c.center_fixed - (i64)y * FIXED_UNIT;
    if (row < 0) row = -row;
    const i64 visibility = min64(mul64_u32(row, (unsigned)glob) >> 16, 24 * FIXED_UNIT);
    const i64 plane_shade = 64 * FIXED_UNIT - ((i64)light + 12) * (FIXED_UNIT / 4);
    const unsigned colormap_row = (unsigned)clampi((plane_shade - visibility) >> 16, 0, 31);
    auto low = [](u64 value) { return (unsigned)value & 0xFFFFFFu; };
    auto high = [](u64 value) { return (unsigned)(value >> 24) & 0xFFFFFFu; };
    PlaneSpan s;
    s.start = make_uint4(low(x), high(x), low(v), high(v));
    s.step = make_uint4(low(xadd) | ((24u - (unsigned)width_bits) << 24), high(xadd) | (colormap_row << 24), low(yadd) | ((24u - (unsigned)height_bits) << 24), high(yadd));
    s.texture = (unsigned)texture * (unsigned)m->tex_max_h * (unsigned)m->tex_max_w;
    return s;
}

// Visplane repair (engine.py:11026-11135) of the noted row ranges.  Every pixel of those rows is selected first (the repairs
// read whole rows and columns).  Vertical: an unresolved pixel takes the sector of the next resolved pixel below it in its
// half of the screen; rows below the noted range are selected until every column that still looks for one has found it.
// Horizontal: an unresolved pixel between a left and a right anchor of one sector takes that sector.  Pixels outside the
// noted rows need none of this: no shown pixel there is unresolved, and resolved pixels are never repaired.
// Every pixel of the noted rows: a wavefront takes 64 columns of a row of the work list at a time, so that lanes with many rows
// and lanes with none load the chip alike.
template <bool MASKS>
__global__ void __launch_bounds__(256) flat_span_select_kernel(DeviceMap dm, gd_lanes_desc lanes, int lane_base, Scratch sc) {
    __shared__ RowLds row_lds[4];
    const int wave = threadIdx.x >> 6, lane_id = threadIdx.x & 63;
    const int total = *sc.flat_row_count * (SW / 64);
    for (int task = blockIdx.x * 4 + wave; task < total; task += gridDim.x * 4) {
        const int entry = task / (SW / 64), x = (task - entry * (SW / 64)) * 64 + lane_id;
        const int packed = sc.flat_rows[entry], local = packed >> 8, y = packed & 255;
        const int s = flat_select_row<MASKS>(dm, sc, lanes, local, lane_base + local, x, y, true, &row_lds[wave]);
        const size_t i = (size_t)local * VH * SW + (size_t)y * SW + x;
        sc.flat_sector[i] = (unsigned short)(s < 0 ? sc.ctx[local].sector : s);
        sc.flat_flags[i] = s < 0 ? 1 : 0;
    }
}

// A column whose pixel in the last noted row of a half is unresolved looks further down for a resolved one
// (engine.py:11026-11083).  A wavefront takes 64 columns of a row at a time, like flat_span_select_kernel; the columns that look no
// further, by what the rows above it have found so far, are left out.  (A work-group of sixteen wavefronts went down 64 columns
// sixteen rows at a time, a step after the other and, for its LDS, one work-group a compute unit: 39 us at 256 lanes of 800
// linedefs, 60 at 512 of 4000, 120 at 1024 of 2000; now 18, 35 and 61.)
template <bool MASKS>
__global__ void __launch_bounds__(256) flat_tail_kernel(DeviceMap dm, gd_lanes_desc lanes, int lane_base, int lane_count, Scratch sc) {
    __shared__ RowLds row_lds[4];
    const int wave = threadIdx.x >> 6, lane_id = threadIdx.x & 63;
    const int total = sc.flat_row_count[1] * (SW / 64);
    for (int task = blockIdx.x * 4 + wave; task < total; task += gridDim.x * 4) {
        const int entry = task / (SW / 64), x = (task - entry * (SW / 64)) * 64 + lane_id;
        const int packed = sc.flat_rows[(size_t)lane_count * VH - 1 - entry], local = packed >> 8, y = packed & 255;
        const int half = y > sc.ctx[local].last_ceiling_row ? 1 : 0, last = sc.flat_span[(size_t)local * 4 + 2 * half + 1];
        unsigned int *found = sc.flat_tail + ((size_t)local * 2 + half) * SW + x;
        const bool looking = (sc.flat_flags[(size_t)local * VH * SW + (size_t)last * SW + x] & 1) &&
                             __hip_atomic_load(found, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) > ((unsigned)y << 16);
        if (__ballot(looking) == 0) continue;
        const int s = flat_select_row<MASKS>(dm, sc, lanes, local, lane_base + local, x, y, looking, &row_lds[wave]);
        if (looking && s >= 0) atomicMin(found, ((unsigned)y << 16) | (unsigned)s);
    }
}

// The repairs of one half of a lane's screen, a work-group per entry of the work list.  The kernel lasts as long as its tallest ranges, whose rows
// depend on each other from the lowest up; so a band of rows is read at once, four columns of FINISH_ROWS rows a thread, and what the
// rows below found travels through LDS in one step.  The rows wait in LDS and not in registers so that only the loads are unrolled: a
// work-group runs through its code once, and what it waits for most is the code.  (A thread a column, eight rows at a time with stores between the
// loads: 62 us for 94 rows of one of 16 lanes, 79 us for 4096 lanes; rows in registers, all loops unrolled, 20 and 40 us; now 14 and 25.)
#define FINISH_QUADS (SW / 4)
#define FINISH_CHUNKS 12          // threads that share four columns
#define FINISH_ROWS 9             // rows a thread takes: a band of 108 rows, the half of a level view
#define FINISH_THREADS (FINISH_QUADS * FINISH_CHUNKS)
#define FINISH_BAND (FINISH_CHUNKS * FINISH_ROWS)
#define FINISH_NONE 0xFFFFu       // no resolved pixel (sectors are below 8191)
__global__ void __launch_bounds__(FINISH_THREADS) flat_span_finish_kernel(Scratch sc) {
    __shared__ uint2 row_sectors[FINISH_ROWS][FINISH_THREADS];
    __shared__ unsigned int row_flags[FINISH_ROWS][FINISH_THREADS];
    __shared__ uint2 topmost[FINISH_CHUNKS][FINISH_QUADS];   // the sectors of four columns' topmost resolved pixels in a thread's rows
    __shared__ unsigned int anchors[FINISH_BAND][SW / 32];   // per row of the band, a bit a column: the pixels that are anchors
    __shared__ unsigned int open[FINISH_BAND][SW / 32];      // likewise: shown, unresolved and no anchors
    const int chunk = threadIdx.x / FINISH_QUADS, quad = threadIdx.x - chunk * FINISH_QUADS, x0 = quad * 4;
    const int total = *sc.flat_span_count;
    auto sector_of = [](const uint2 &four, int k) { return ((k < 2 ? four.x : four.y) >> (16 * (k & 1))) & 0xFFFFu; };
    for (int entry = blockIdx.x; entry < total; entry += gridDim.x) {
        const int packed = sc.flat_spans[entry], local = packed >> 1, half = packed & 1;
        const int lo = sc.flat_span[(size_t)local * 4 + 2 * half], hi = sc.flat_span[(size_t)local * 4 + 2 * half + 1];
        const unsigned camera_sector = (unsigned)sc.ctx[local].sector;
        unsigned short *sector = sc.flat_sector + (size_t)local * VH * SW;
        unsigned char *flags = sc.flat_flags + (size_t)local * VH * SW;
        const unsigned int *meta = sc.meta + (size_t)local * VH * SW;
        // what flat_tail_kernel found below the range for a column whose pixel in the range's last row is unresolved
        const uint4 tail = *reinterpret_cast<const uint4 *>(sc.flat_tail + ((size_t)local * 2 + half) * SW + x0);
        unsigned below[4] = {tail.x & 0xFFFFu, tail.y & 0xFFFFu, tail.z & 0xFFFFu, tail.w & 0xFFFFu};
        for (int band_hi = hi; band_hi >= lo; band_hi -= FINISH_BAND) {
            const int rows = min(band_hi - lo + 1, FINISH_BAND), band_lo = band_hi - rows + 1;
            const int each = (rows + FINISH_CHUNKS - 1) / FINISH_CHUNKS, first = band_hi - chunk * each;   // a thread's rows, the lowest first
            const int own = max(min(each, first - band_lo + 1), 0);
            unsigned int flags_read[FINISH_ROWS]; uint2 sectors_read[FINISH_ROWS]; uint4 words[FINISH_ROWS];
#pragma unroll
            for (int j = 0; j < FINISH_ROWS; ++j) {   // rows past the thread's own are read again and left out below
                const size_t i = (size_t)max(first - min(j, each - 1), band_lo) * SW + x0;
                flags_read[j] = *reinterpret_cast<const unsigned int *>(flags + i);
                sectors_read[j] = *reinterpret_cast<const uint2 *>(sector + i);
                words[j] = *reinterpret_cast<const uint4 *>(meta + i);
            }
            __syncthreads();                          // nobody reads the previous band's anchors and topmost pixels any more
            u64 shown = 0;                            // a bit a pixel: does it show the flat pass's picture?
#pragma unroll
            for (int j = 0; j < FINISH_ROWS; ++j) {
                row_flags[j][threadIdx.x] = flags_read[j]; row_sectors[j][threadIdx.x] = sectors_read[j];
                const unsigned gap = (gap_pixel(words[j].x) ? 1u : 0u) | (gap_pixel(words[j].y) ? 2u : 0u) | (gap_pixel(words[j].z) ? 4u : 0u) | (gap_pixel(words[j].w) ? 8u : 0u);
                shown |= (u64)gap << (4 * j);
            }
            for (int k = threadIdx.x; k < rows * (SW / 32); k += FINISH_THREADS) { (&anchors[0][0])[k] = 0u; (&open[0][0])[k] = 0u; }
            unsigned span_sector[4] = {FINISH_NONE, FINISH_NONE, FINISH_NONE, FINISH_NONE};
#pragma unroll 1
            for (int j = 0; j < own; ++j) {
                const unsigned int four = row_flags[j][threadIdx.x];
                const uint2 sectors = row_sectors[j][threadIdx.x];
#pragma unroll
                for (int k = 0; k < 4; ++k) span_sector[k] = (four >> (8 * k)) & 1u ? span_sector[k] : sector_of(sectors, k);
            }
            topmost[chunk][quad] = make_uint2(span_sector[0] | (span_sector[1] << 16), span_sector[2] | (span_sector[3] << 16));
            __syncthreads();
            // --- vertical (engine.py:11026-11083): floors and ceilings alike look downwards, within their own half
#pragma unroll 1
            for (int c = 0; c < FINISH_CHUNKS; ++c) {
                const uint2 four = topmost[c][quad];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    span_sector[k] = c <= chunk ? below[k] : span_sector[k];   // what lies below the thread's own rows
                    below[k] = sector_of(four, k) != FINISH_NONE ? sector_of(four, k) : below[k];
                }
            }
#pragma unroll 1
            for (int j = 0; j < own; ++j) {
                const unsigned int four = row_flags[j][threadIdx.x];
                const uint2 sectors = row_sectors[j][threadIdx.x];
                unsigned int anchor = 0u, new_flags = four, pair[2] = {sectors.x, sectors.y};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const bool resolved = !((four >> (8 * k)) & 1u);
                    if (resolved) span_sector[k] = sector_of(sectors, k);
                    const bool found = span_sector[k] != FINISH_NONE, anchors_here = resolved || (found && span_sector[k] != camera_sector);
                    if (!resolved && found) {
                        pair[k >> 1] = (pair[k >> 1] & ~(0xFFFFu << (16 * (k & 1)))) | (span_sector[k] << (16 * (k & 1)));
                        // bit1: vertical span; bit2: its sector differs from the camera's (anchor)
                        new_flags |= (2u | (anchors_here ? 4u : 0u)) << (8 * k);
                    }
                    anchor |= anchors_here ? 1u << k : 0u;
                }
                if (new_flags != four) {
                    const size_t i = (size_t)(first - j) * SW + x0;
                    *reinterpret_cast<unsigned int *>(flags + i) = new_flags;
                    *reinterpret_cast<uint2 *>(sector + i) = make_uint2(pair[0], pair[1]);
                    row_flags[j][threadIdx.x] = new_flags; row_sectors[j][threadIdx.x] = make_uint2(pair[0], pair[1]);
                }
                const unsigned int wants = ~anchor & (unsigned)(shown >> (4 * j)) & 15u;
                if (anchor) atomicOr(&anchors[first - j - band_lo][quad >> 3], anchor << (4 * (quad & 7)));
                if (wants) atomicOr(&open[first - j - band_lo][quad >> 3], wants << (4 * (quad & 7)));
            }
            __syncthreads();
            // --- horizontal (engine.py:11085-11135): a shown pixel between a left and a right anchor of one sector.  (An anchor is
            // its own on either side; what is not shown needs no repair.)  A thread a word of 32 columns: the pixels are mostly one below the other.
            for (int task = threadIdx.x; task < rows * (SW / 32); task += FINISH_THREADS) {
                const int row = task / (SW / 32), word = task - row * (SW / 32), from_low = rows - 1 - row, holder = from_low / each, j = from_low - holder * each;
                const unsigned int *row_anchors = anchors[row];
                for (unsigned int rest = open[row][word]; rest; rest &= rest - 1u) {
                    const int bit = __ffs((int)rest) - 1;
                    int left = -1, right = SW;        // this pixel is no anchor: the nearest ones on either side
                    for (int w = word; w >= 0 && left < 0; --w) {
                        const unsigned int bits = row_anchors[w] & (w == word ? (1u << bit) - 1u : ~0u);
                        if (bits) left = w * 32 + 31 - __clz((int)bits);
                    }
                    for (int w = word; w < SW / 32 && right >= SW; ++w) {
                        const unsigned int bits = row_anchors[w] & (w == word ? ~0u << bit : ~0u);
                        if (bits) right = w * 32 + __ffs((int)bits) - 1;
                    }
                    if (left < 0 || right >= SW) continue;
                    const uint2 *held = &row_sectors[j][holder * FINISH_QUADS];      // anchors are not rewritten here
                    const unsigned left_sector = sector_of(held[left >> 2], left & 3), right_sector = sector_of(held[right >> 2], right & 3);
                    if (left_sector != right_sector) continue;
                    const int x = word * 32 + bit;
                    const size_t i = (size_t)(band_lo + row) * SW + x;
                    sector[i] = (unsigned short)left_sector;
                    flags[i] = (unsigned char)(((row_flags[j][holder * FINISH_QUADS + (x >> 2)] >> (8 * (x & 3))) & 0xFFu) | 8u);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// walls: engine.py:11462-13745
// ---------------------------------------------------------------------------------------------
struct ColumnCtx {
    const Tables *tb;
    const gd_map_desc *m;
    MapView mv;
    const LaneCtx *c;
    const WallRec *recs;  // the chunk's [L,W] records, with rec_base = lane * W
    const RecSpan *spans; // the chunk's [L,W] ray-test facts of every linedef
    const WallRec *frags; // this lane's [split_count, fragment_slots] fragment records
    const Cand *list;     // the chunk's candidate blocks; entry k of this column sits list_column + k * 320 * 8 bytes in
    unsigned rec_base, list_column;
    int count;
    int x;
    float rx, ry;
    Eval first;           // linedef 0 at this column, which stands in where a pass finds none
    __device__ __forceinline__ const WallRec &rec(int w) const { return recs[rec_base + (unsigned)w]; }
    // Where the list of column `x` of the chunk's lane `local` starts and how many entries it has: the column's own
    // slots, or its slot in the spill pool.
    __device__ __forceinline__ void set_list(const Scratch &sc, int local, int column) {
        list = sc.cand;
        const int listed = sc.cand_count[(size_t)local * SW + column];
        const unsigned spill = (unsigned)listed >> SPILL_SHIFT;
        if (spill) {
            const unsigned slot = spill - 1;
            list_column = (sc.spill_base + (slot / SW) * (unsigned)(SPILL_DEPTH * SW) + slot % SW) * 8u;
            count = listed & ((1 << SPILL_SHIFT) - 1);
        } else {
            list_column = ((unsigned)local * (CAND_MAX * SW) + (unsigned)column) * 8u;
            count = listed < CAND_MAX ? listed : CAND_MAX;
        }
    }
    __device__ __forceinline__ u64 cand(int k) const {      // as its key
        return *reinterpret_cast<const u64 *>(reinterpret_cast<const char *>(list) + (list_column + (unsigned)k * (SW * 8u)));
    }
    __device__ Eval eval(int w) const { return eval_wall(m, *c, spans + rec_base, x, w, rx, ry); }
};

#define STANDS_IN (CF_ONE_SIDED | CF_PROJ | CF_LEDGE | CF_SECTOR0)    // all of them: what a column without a sector may find (select_columns)
// A candidate as a scan looks at it.
struct ListEntry {
    unsigned short flags, wall;
    float dist;
    unsigned sectors, vertices;    // as in WallLinks
    __device__ __forceinline__ u64 key() const { return ((u64)__float_as_uint(dist) << 32) | ((u64)wall << 16) | (u64)flags; }
};
// A column's list as wall_select_kernel's LANES lanes of the column hold it between them: entry k in registers of lane k % LANES.  Each
// looks at its own in a scan, and what the scan is after, the smallest of some keys, is exchanged.  One lane alone keeps what is near of it.
template <int LANES> struct ListShare {
    static constexpr int ENTRIES = CAND_MAX / LANES;
    ListEntry own[ENTRIES];
    // an entry that is not there lies nearer than any distance a scan asks for: none takes it
    __device__ __forceinline__ void load(const ColumnCtx &cc, int lane) {
        u64 keys[ENTRIES];
#pragma unroll
        for (int j = 0; j < ENTRIES; ++j) keys[j] = cc.cand(max(min(j * LANES + lane, cc.count - 1), 0));
#pragma unroll
        for (int j = 0; j < ENTRIES; ++j) {
            const bool there = j * LANES + lane < cc.count;
            const Cand q = key_cand(keys[j]);
            const WallLinks &links = cc.mv.walls[there ? q.wall : 0];
            own[j].wall = q.wall; own[j].sectors = links.sectors; own[j].vertices = links.vertices;
            own[j].dist = there ? q.dist : -GD_INF; own[j].flags = there ? q.flags : 0;
        }
    }
    // the smallest of the column's lanes; all of them are executing
    template <int CONTROL> static __device__ __forceinline__ u64 moved(u64 v) {
        return ((u64)(unsigned)__builtin_amdgcn_mov_dpp((int)(v >> 32), CONTROL, 0xF, 0xF, true) << 32) | (u64)(unsigned)__builtin_amdgcn_mov_dpp((int)(v & 0xFFFFFFFFu), CONTROL, 0xF, 0xF, true);
    }
    static __device__ __forceinline__ u64 smallest(u64 v) {
        u64 o;
        if (LANES >= 2) { o = moved<0xB1>(v); v = o < v ? o : v; }      // lanes 1,0,3,2
        if (LANES >= 4) { o = moved<0x4E>(v); v = o < v ? o : v; }      // lanes 2,3,0,1
        if (LANES >= 8) { o = moved<0x141>(v); v = o < v ? o : v; }     // the eight lanes mirrored
        if (LANES >= 16) { o = moved<0x140>(v); v = o < v ? o : v; }    // the sixteen lanes mirrored
        if (LANES >= 32) { o = ((u64)(unsigned)__builtin_amdgcn_ds_swizzle((int)(v >> 32), 0x401F) << 32) | (u64)(unsigned)__builtin_amdgcn_ds_swizzle((int)(v & 0xFFFFFFFFu), 0x401F); v = o < v ? o : v; }
        return v;
    }
    static __device__ __forceinline__ unsigned smallest(unsigned v) {
        if (LANES >= 2) v = min(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true));
        if (LANES >= 4) v = min(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true));
        if (LANES >= 8) v = min(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, true));
        if (LANES >= 16) v = min(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xF, 0xF, true));
        if (LANES >= 32) v = min(v, (unsigned)__builtin_amdgcn_ds_swizzle((int)v, 0x401F));
        return v;
    }
    // every entry of the column that this lane looks at
    template <typename Look> __device__ __forceinline__ void each(const ColumnCtx &cc, Look look) const {
#pragma unroll
        for (int j = 0; j < ENTRIES; ++j) look(own[j]);
    }
};
// The nearest of the candidates a scan takes, the lowest linedef on ties, and its flags.
template <int LANES> struct NearestOf {
    u64 key = CAND_KEY_NONE;
    __device__ __forceinline__ void take(const ListEntry &q) { const u64 k = q.key(); key = k < key ? k : key; }
    __device__ __forceinline__ void share() { key = ListShare<LANES>::smallest(key); }     // what the column's lanes took
    __device__ __forceinline__ float distance() const { return cand_key_distance(key); }
    __device__ __forceinline__ int wall() const { return cand_key_wall(key); }
    __device__ __forceinline__ int flags() const { return cand_key_flags(key); }
};
template <> struct NearestOf<1> {
    float d = GD_INF; int w = 0x7fffffff, f = 0;
    __device__ __forceinline__ void take(const ListEntry &q) { if (q.dist < d || (q.dist == d && (int)q.wall < w)) { d = q.dist; w = q.wall; f = q.flags; } }
    __device__ __forceinline__ void share() {}
    __device__ __forceinline__ float distance() const { return d; }
    __device__ __forceinline__ int wall() const { return w; }
    __device__ __forceinline__ int flags() const { return f; }
};
// One lane alone keeps the nearest entries beyond the column's distance in LDS, in order, with their sectors: the window.  A scan goes through it until what is
// left is too far to matter, and through the whole list in memory if the window ends before that.  When one of the wavefront's columns has passed
// WINDOW_REFILL entries by, all of them fill theirs again: columns that did so one by one would have the wavefront fill in nearly every pass.
// The launch for all but the longest strips waits for memory more than for anything else (60 % of its wavefronts' time), and the list is what it waited for: 30 KB a
// wavefront at 16 bytes an entry, four times what L2 holds of it.  Read whole by every scan it takes 0.895 ms for 4096 lanes on the 4000-linedef map; only the
// entries' order in LDS, nearest first, 0.79, with as many wavefronts a SIMD as one likes; this way 0.64 (11 million lines missed in L2, 15, 6).  1024 lanes on the
// 2000-linedef map 231, 191, 156 us.  Filled again after 3 / 4 / 5 / 6 / 8 / 10 entries 645 / 646 / 642 / 710 / 730 / 770 us.  Twelve entries are what sixteen
// wavefronts' LDS holds; with sixteen, and eight wavefronts, 1.0 ms.  (All of it before a linedef's record lay in registers, see WallLinks, which made 0.64 ms 0.54.)
#define WINDOW 12
#define WINDOW_REFILL 5
#define WINDOW_BATCH 16        // entries ordered at a time
#define WINDOW_PAD (WINDOW_WALK_ROWS - 1)   // rows read with the last ones: words of other lanes, which window_walk says are not there
template <> struct ListShare<1> {
    static constexpr int WORDS = (WINDOW * 3 + WINDOW_PAD) * 64;
    u64 *keys;                  // this lane's word of [WINDOW][64]
    unsigned *sectors;          // the same of theirs, behind the keys
    u64 solid_ledges, ledges;   // bit k: the entries k, k + 64, ... hold one whose projected span begins at this column (CF_PROJ and CF_LEDGE), one-sided, two-sided
    int from, held;             // the window's entries before `from` are no farther than `passed`; it holds `held`
    float passed, floor;        // floor: `passed` when it was filled
    bool complete;              // nothing of the list lies beyond the window
    static __device__ __forceinline__ u64 smallest(u64 v) { return v; }
    static __device__ __forceinline__ unsigned smallest(unsigned v) { return v; }

    __device__ __forceinline__ void start(const ColumnCtx &cc, unsigned *words, int lane_id, bool &any_ledge, bool &stand_in) {
        keys = reinterpret_cast<u64 *>(words) + lane_id; sectors = words + WINDOW * 2 * 64 + lane_id;
        solid_ledges = 0; ledges = 0; from = 0; held = 0; passed = 0.0f; floor = GD_INF; complete = false;
        unsigned flagged = 0;
        for (int k0 = 0; k0 < cc.count; k0 += 8) {
            unsigned flags[8], solid = 0, portal = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) flags[j] = (unsigned)cc.cand(k0 + j);     // what lies behind the list's end is memory of the column's all the same
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const unsigned f = k0 + j < cc.count ? flags[j] : 0u;
                flagged |= f;
                const bool ledge = (f & (CF_LEDGE | CF_PROJ)) == (CF_LEDGE | CF_PROJ);
                solid |= ledge && (f & CF_ONE_SIDED) ? 1u << j : 0u;
                portal |= ledge && !(f & CF_ONE_SIDED) ? 1u << j : 0u;
                stand_in |= (f & STANDS_IN) == STANDS_IN;
            }
            solid_ledges |= (u64)solid << (k0 & 63);
            ledges |= (u64)portal << (k0 & 63);
        }
        any_ledge = flagged & CF_LEDGE;
    }
    // The window: the nearest entries beyond `passed`.  Keys are positive float64 numbers (a float32's exponent of all ones is not one of float64's), whose
    // order is theirs: an exchange is a minimum and a maximum.
    __device__ __forceinline__ void fill(const ColumnCtx &cc) {
        double best[WINDOW_BATCH];
        const double none = __longlong_as_double((long long)CAND_KEY_NONE);
        int beyond = 0;
#pragma unroll
        for (int j = 0; j < WINDOW_BATCH; ++j) best[j] = none;
        for (int k0 = 0; k0 < cc.count; k0 += WINDOW_BATCH) {
            u64 raw[WINDOW_BATCH];
            double next[WINDOW_BATCH];
#pragma unroll
            for (int j = 0; j < WINDOW_BATCH; ++j) raw[j] = cc.cand(k0 + j);
#pragma unroll
            for (int j = 0; j < WINDOW_BATCH; ++j) {
                const bool wanted = k0 + j < cc.count && cand_key_distance(raw[j]) > passed;
                beyond += wanted ? 1 : 0;
                next[j] = wanted ? __longlong_as_double((long long)raw[j]) : none;
            }
            order_up(next);
            if (k0 == 0) {
#pragma unroll
                for (int j = 0; j < WINDOW_BATCH; ++j) best[j] = next[j];
            } else {
                order_merge_lowest(best, next);
            }
        }
        held = min(beyond, WINDOW); complete = beyond <= WINDOW;
        from = 0; floor = passed;
        unsigned pairs[WINDOW];
#pragma unroll
        for (int j = 0; j < WINDOW; ++j) {
            const u64 key = (u64)__double_as_longlong(best[j]);
            pairs[j] = cc.mv.walls[key == CAND_KEY_NONE ? 0 : (unsigned)key >> 16].sectors;
            keys[j * 64] = key;
        }
#pragma unroll
        for (int j = 0; j < WINDOW; ++j) sectors[j * 64] = pairs[j];
    }
    // A pass of the column begins: its scans ask for entries beyond `distance`.
    __device__ __forceinline__ void begin(const ColumnCtx &cc, float distance) {
        passed = distance;
        if (__ballot(distance < floor || (from >= WINDOW_REFILL && !complete)) != 0 && !(complete && distance >= floor)) fill(cc);
    }
    // The entries beyond `passed` (and some that are not, and some twice), nearest first as far as the window goes, until those left are
    // farther than enough().
    template <bool ADVANCE, typename Look, typename Enough> __device__ __forceinline__ void walk(const ColumnCtx &cc, Look look, Enough enough) {
        auto row = [&](int k) { const Cand q = key_cand(keys[k * 64]); return ListEntry{q.flags, q.wall, q.dist, sectors[k * 64], 0u}; };
        const bool ended = window_walk<ADVANCE>(from, held, passed, row, look, enough);
        if (complete || ended) return;
        for (int k0 = 0; k0 < cc.count; k0 += 4) {
            u64 key[4]; unsigned pair[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) key[j] = cc.cand(k0 + j);
#pragma unroll
            for (int j = 0; j < 4; ++j) pair[j] = cc.mv.walls[k0 + j < cc.count ? (unsigned)key[j] >> 16 : 0u].sectors;
#pragma unroll
            for (int j = 0; j < 4; ++j) { const Cand q = key_cand(key[j]); look(ListEntry{q.flags, q.wall, q.dist, pair[j], 0u}, k0 + j < cc.count); }
        }
    }
    template <typename Look> __device__ __forceinline__ void each_of(const ColumnCtx &cc, u64 places, Look look) const {
        for (u64 rest = places; rest; rest &= rest - 1)
            for (int k = __ffsll((long long)rest) - 1; k < cc.count; k += 64) {
                const Cand q = key_cand(cc.cand(k));
                const WallLinks &links = cc.mv.walls[q.wall];
                look(ListEntry{q.flags, q.wall, q.dist, links.sectors, links.vertices});
            }
    }
};

// The projection fragment of a linedef at one column (engine.py:11511-11529, 12324-12376): the first
// present fragment whose half-open span holds the column.  A linedef that was never split is its own
// fragment.  `has` is false where no fragment holds the column (OWallMost then falls back to the whole
// linedef, engine.py:12598-12604); `lights` tells whether wallscan light interpolates over the fragment,
// which only linedefs with several fragments do (engine.py:11530-11545).
struct FragmentChoice {
    const WallRec *rec;
    bool has, lights;
};
// SPLIT is false for maps without split linedefs, whose kernels then carry none of the search.
template <bool SPLIT>
__device__ __forceinline__ FragmentChoice choose_fragment(const gd_map_desc *m, const WallRec *frags, const WallRec &whole, int w, int x) {
    FragmentChoice f;
    f.rec = &whole; f.lights = false;
    f.has = (whole.sr > whole.sl) && (x >= whole.sl) && (x < whole.sr);
    if (SPLIT && (whole.flags & WF_SPLIT)) {
        const int F = m->fragment_slots, row = m->wall_split_slot[w];
        int count = 0;
        f.has = false;
        for (int k = 0; k < F; ++k) {
            if (!m->split_fragment_mask[row * F + k]) continue;
            ++count;
            const WallRec &g = frags[row * F + k];
            if (!f.has && (g.sr > g.sl) && (x >= g.sl) && (x < g.sr)) { f.rec = &g; f.has = true; }
        }
        f.lights = f.has && count > 1;
        if (!f.has) f.rec = &whole;
    }
    return f;
}

// engine.py:11217-11291 for one endpoint order, evaluated at one column
__device__ i64 wall_visibility(const WallRec &r, int side, int x) {
    i64 tx1 = side ? r.tx1 : r.tx0, tx2 = side ? r.tx0 : r.tx1;
    i64 ty1 = side ? r.ty1 : r.ty0, ty2 = side ? r.ty0 : r.ty1;
    const i64 center = 160 * FIXED_UNIT;
    i64 safe_ty1 = ty1 == 0 ? 1 : ty1, safe_ty2 = ty2 == 0 ? 1 : ty2;
    i64 left_projected = ((center + tdiv(tx1 * center, safe_ty1)) >> 16) + (tx1 >= 0);
    i64 right_projected = ((center + tdiv(tx2 * center, safe_ty2)) >> 16) + (tx2 >= 0);
    i64 left_den = tx1 - tx2 - ty2 + ty1, right_den = ty2 - ty1 - tx2 + tx1;
    i64 safe_left_den = left_den == 0 ? 1 : left_den, safe_right_den = right_den == 0 ? 1 : right_den;
    bool left_inside = tx1 >= -ty1, right_inside = tx2 <= ty2;
    i64 wsl = left_inside ? left_projected : 0;
    i64 wsr = right_inside ? right_projected : SW;
    i64 wdl = left_inside ? ty1 : ty1 + tdiv((ty2 - ty1) * (tx1 + ty1), safe_left_den);
    i64 wdr = right_inside ? ty2 : ty1 + tdiv((ty2 - ty1) * (tx1 - ty1), safe_right_den);
    i64 light_left = tdiv(WALL_VISIBILITY_FIXED << 12, max64(wdl, 1));
    i64 light_right = tdiv(WALL_VISIBILITY_FIXED << 12, max64(wdr, 1));
    i64 light_step = tdiv(light_right - light_left, max64(wsr - wsl, 1));
    return light_left + ((i64)x - wsl) * light_step;
}

// engine.py:10672-10739 (PrepWall) for one (linedef, column)
// `ends`: anything with the linedef's view-space endpoints (WallRec, WallGeo)
template <typename Ends>
__device__ __forceinline__ void texture_mapping(const Ends &ends, i64 linedef_repeat, int x, i64 *hoff, i64 *vstep) {
    const float wall_map_scale = (float)((320 * 200.0 / 320.0 / 240) * 64.0 / (320 / 2.0));
    i64 tx1 = ends.tx0, tx2 = ends.tx1, ty1 = ends.ty0, ty2 = ends.ty1;
    double u_over_z_origin = (double)((float)tx1 * 160.0f);
    float u_over_z_step_f = -(float)ty1;
    double u_over_z_step = (double)u_over_z_step_f;
    double inv_z_origin = (double)((float)(tx1 - tx2) * 160.0f);
    float inv_z_step_float = (float)(ty2 - ty1);
    double inv_z_step = (double)inv_z_step_float;
    double depth_scale = (double)(inv_z_step_float * wall_map_scale);
    double depth_origin = (double)(-u_over_z_step_f * wall_map_scale);
    double repeat = (double)linedef_repeat;
    double column = (double)x - 160.0;
    double top = u_over_z_origin + u_over_z_step * column;
    double bottom = inv_z_origin + inv_z_step * column;
    double safe_bottom = bottom == 0 ? 1.0 : bottom;
    double fraction = top / safe_bottom;
    *hoff = f64_to_i64(floor(fraction * repeat + 0.5));
    *vstep = f64_to_i64(floor(fraction * depth_scale + depth_origin + 0.5));
}

// engine.py:12294-12605 (OWallMost) for one column
__device__ __forceinline__ float project(const LaneCtx &c, const WallRec &g, const FragmentChoice &fragment, float world_z, int x) {
    i64 whole_sl = g.sl, whole_sr = g.sr;
    i64 whole_dl = max64(g.dl, 1), whole_dr = max64(g.dr, 1);
    const bool has_fragment = fragment.has;
    const WallRec &f = *fragment.rec;
    i64 screen_left = f.sl, screen_right = f.sr, depth_left = max64(f.dl, 1), depth_right = max64(f.dr, 1);
    i64 relative_z_fixed = round_to_i64((world_z - c.view_z) * 65536.0f);
    i64 pz = -(relative_z_fixed >> 4);
    i64 center_fixed = c.center_fixed;
    i64 px = x;
    if (!has_fragment) {
        i64 original_span = max64(whole_sr - whole_sl, 1);
        i64 opl = tdiv(mul64(pz, FOCAL_Y_FIXED), whole_dl);
        i64 opr = tdiv(mul64(pz, FOCAL_Y_FIXED), whole_dr);
        i64 ostep = tdiv(opr - opl, original_span);
        return (float)clampi((center_fixed + opl + mul64(px - whole_sl, ostep)) >> 16, 0, VH);
    }
    const i64 upper_clip = c.upper_clip, lower_clip = c.lower_clip;
    i64 upper_left = mul64(upper_clip, depth_left) >> 16, upper_right = mul64(upper_clip, depth_right) >> 16;
    i64 lower_left = mul64(lower_clip, depth_left) >> 16, lower_right = mul64(lower_clip, depth_right) >> 16;
    bool above_left = pz < upper_left, above_right = pz < upper_right;
    bool below_left = pz > lower_left, below_right = pz > lower_right;
    bool entirely_above = above_left && above_right, entirely_below = below_left && below_right;
    i64 clipped_left = screen_left, clipped_right = screen_right;
    i64 clipped_dl = depth_left, clipped_dr = depth_right;
    bool outside_top = false, outside_bottom = false;
    bool crosses_top = above_left != above_right;
    if (crosses_top) {
        i64 safe_upper_delta = (upper_right != upper_left) ? (upper_right - upper_left) : 1;
        i64 top_fraction = tdiv(shl64(pz - upper_left, 30), safe_upper_delta);
        i64 top_depth = depth_left + (mul64(depth_right - depth_left, top_fraction) >> 30);
        i64 top_cross = screen_left + tdiv(mul64(mul64(depth_right, top_fraction) >> 30, screen_right - screen_left), max64(top_depth, 1));
        if (above_right && (screen_left <= top_cross)) { clipped_right = top_cross; clipped_dr = top_depth; }
        outside_top |= above_right && (screen_right > top_cross) && (px >= top_cross) && (px < screen_right);
        if (above_left && (top_cross <= screen_right)) { clipped_left = top_cross; clipped_dl = top_depth; }
        outside_top |= above_left && (top_cross > screen_left) && (px >= screen_left) && (px < top_cross);
    }
    bool crosses_bottom = below_left != below_right;
    if (crosses_bottom) {
        i64 safe_lower_delta = (lower_right != lower_left) ? (lower_right - lower_left) : 1;
        i64 bottom_fraction = tdiv(shl64(pz - lower_left, 30), safe_lower_delta);
        i64 bottom_depth = depth_left + (mul64(depth_right - depth_left, bottom_fraction) >> 30);
        i64 bottom_cross = screen_left + tdiv(mul64(mul64(depth_right, bottom_fraction) >> 30, screen_right - screen_left), max64(bottom_depth, 1));
        if (below_right && (screen_left <= bottom_cross)) { clipped_right = bottom_cross; clipped_dr = bottom_depth; }
        outside_bottom |= below_right && (screen_right > bottom_cross) && (px >= bottom_cross) && (px < screen_right);
        if (below_left && (bottom_cross <= screen_right)) { clipped_left = bottom_cross; clipped_dl = bottom_depth; }
        outside_bottom |= below_left && (bottom_cross > screen_left) && (px >= screen_left) && (px < bottom_cross);
    }
    i64 projected_left = tdiv(mul64(pz, FOCAL_Y_FIXED), max64(clipped_dl, 1));
    i64 projected_right = tdiv(mul64(pz, FOCAL_Y_FIXED), max64(clipped_dr, 1));
    i64 span = max64(clipped_right - clipped_left, 1);
    i64 projected_step = tdiv(projected_right - projected_left, span);
    i64 projected = clampi((center_fixed + projected_left + mul64(px - clipped_left, projected_step)) >> 16, 0, VH);
    bool collapsed = (clipped_right == clipped_left) && (px == clipped_left) && !(entirely_above || entirely_below);
    if (entirely_above || (outside_top && !collapsed)) projected = 0;
    else if (entirely_below || (outside_bottom && !collapsed)) projected = VH;
    return (float)projected;
}

// engine.py:10630-10640
__device__ __forceinline__ i64 wall_shade(float light, i64 visibility) {
    i64 shade = 64 * FIXED_UNIT - ((i64)light + 12) * (FIXED_UNIT / 4);
    return clampi((shade - min64(visibility, 24 * FIXED_UNIT)) >> 16, 0, 31);
}

// engine.py:11596-11730 for one (column, linedef): the owner and, if that is another linedef, what its ray test says
__device__ __forceinline__ void endpoint_owner(const ColumnCtx &cc, int w, const Eval &cw, const WallLinks &links, int *owner_index, Eval *owner) {
    const gd_map_desc *m = cc.m;
    const int K = m->neighbor_slots;
    const bool subpixel = cw.flags & CF_SUBPIXEL;
    float tol_w = tolerance_of(cw.dist);
    *owner_index = w; *owner = cw;
    // the owner only matters for a linedef that does not own this column itself (engine.py:11716)
    if (cw.flags & CF_PROJ) return;
    bool uses_start = !(cw.flags & CF_ALONG_HI);
    int index; Eval found; bool valid;
    if (m->direct_neighbors) {
        // slots: start slot | end slot << 8 | has start << 16 | has end << 17
        int ss = links.slots & 0xFF, es = (links.slots >> 8) & 0xFF; bool hs = (links.slots >> 16) & 1, he = (links.slots >> 17) & 1;
        int rslot = uses_start ? ss : es, oslot = uses_start ? es : ss;
        bool rexists = uses_start ? hs : he, oexists = uses_start ? he : hs;
        const int at_start = links.neighbour[0], at_end = links.neighbour[1];      // values: see WallLinks
        int rn = uses_start ? at_start : at_end, on = uses_start ? at_end : at_start;
        Eval r = cc.eval(rn);
        bool r_owns = rexists && (r.flags & CF_PROJ) && (r.flags & CF_LEDGE);
        index = rn; found = r; valid = r_owns;
        if (subpixel && oexists) {
            Eval o = cc.eval(on);
            bool o_owns = (o.flags & CF_PROJ) && (o.flags & CF_LEDGE) && (fabsf(o.dist - cw.dist) <= tol_w);
            if (o_owns && (!r_owns || (o.dist < r.dist) || ((o.dist == r.dist) && (oslot < rslot)))) { index = on; found = o; }
            valid = r_owns || o_owns;
        }
    } else {
        float best = GD_INF; int best_slot = 0;
        for (int k = 0; k < K; ++k) {
            int n = m->endpoint_neighbors[w * K + k];
            bool st = m->endpoint_neighbor_starts[w * K + k], en = m->endpoint_neighbor_ends[w * K + k];
            Eval nb = cc.eval(n);
            bool ray_nb = uses_start ? st : en;
            bool selected = ray_nb || (subpixel && (st || en) && (fabsf(nb.dist - cw.dist) <= tol_w));
            float v = ((nb.flags & CF_PROJ) && (nb.flags & CF_LEDGE) && selected) ? nb.dist : GD_INF;
            if (v < best) { best = v; best_slot = k; }
        }
        index = m->endpoint_neighbors[w * K + best_slot];
        valid = finitef(best);
        if (valid) found = cc.eval(index);
    }
    if (valid) { *owner_index = index; *owner = found; }
}


struct ColumnState {   // engine.py:11561-11580, 11735-11762
    int current_sector;
    float ceiling_clip, floor_clip;
    float masked_ceiling_clip, masked_floor_clip, masked_distance;
    int masked_wall;
    float previous_distance;
    int pend_po_vertex, pend_ep_vertex, pend_ep_wall, pend_eb_index, pend_pb_index, pend_pb_sector;
    float pend_pb_exit;
    unsigned pend_ep_sectors, pend_ep_vertices;   // pend_ep_wall's
    int flags;  // bit0 pend_po_boundary, bit1 pend_ep_boundary, bit2 pend_eb_boundary, bit3 pend_pb
};
#define ST_PO 1
#define ST_EP 2
#define ST_EB 4
#define ST_PB 8

__device__ __forceinline__ bool same_state(const ColumnState &a, const ColumnState &b) {
    return a.current_sector == b.current_sector && a.ceiling_clip == b.ceiling_clip && a.floor_clip == b.floor_clip &&
           a.masked_ceiling_clip == b.masked_ceiling_clip && a.masked_floor_clip == b.masked_floor_clip &&
           a.masked_distance == b.masked_distance && a.masked_wall == b.masked_wall &&
           a.previous_distance == b.previous_distance && a.pend_po_vertex == b.pend_po_vertex &&
           a.pend_ep_vertex == b.pend_ep_vertex && a.pend_ep_wall == b.pend_ep_wall && a.pend_eb_index == b.pend_eb_index &&
           a.pend_pb_index == b.pend_pb_index && a.pend_pb_sector == b.pend_pb_sector && a.pend_pb_exit == b.pend_pb_exit &&
           a.flags == b.flags;
}

struct PassColumn {
    int wall, side, render_current, other_sector;
    float distance;
    int ps_path_index, ps_other, no_path_other, sel_vertex, fb_idx;
    float ps_path_distance, no_path_distance;
    unsigned sectors, vertices;   // wall's
    int bits, marks;       // PB_*, REC_*
};
#define PB_VALID 0x1
#define PB_RASTER 0x2
#define PB_ONE_SIDED 0x4
#define PB_PS_KEEPS 0x100
#define PB_NO_KEEPS 0x200
#define PB_GEOMETRIC 0x400
#define PB_REPLACE_NP 0x800
#define PB_PS_FROM_FRONT 0x1000
#define PB_CONTINUES_PO 0x2000
#define PB_FORWARD_BRIDGE 0x4000
#define PB_FINAL_ALONG_HI 0x8000

__device__ __forceinline__ float height_row(const ColumnLine &line, int x) { return (float)(int)clampi(line.at(x) >> 16, 0, VH); }
__device__ __forceinline__ float bent_row(float row, const HeightBend &b, int x) {
    const int top0 = b.top & 1023u, top1 = (b.top >> 10) & 1023u, collapsed = (int)(b.top >> 20) - 1;
    const int bottom0 = b.bottom & 1023u, bottom1 = (b.bottom >> 10) & 1023u;
    if (x >= bottom0 && x < bottom1 && x != collapsed) row = (float)VH;
    if (x >= top0 && x < top1 && x != collapsed) row = 0.0f;
    return row;
}
__device__ __forceinline__ bool bends(const HeightBend &b) { return (b.bottom >> 31) != 0; }

// The rows of a linedef's four heights at column x: ceiling and floor of the sector its front (`back`: its back) side faces, floor
// and ceiling of the other one.  Nothing here waits for a load before the next is asked for, except in columns
// outside the span of a linedef with a height that bends, which are few.
struct WallRows { float ceiling, floor, other_floor, other_ceiling; };
__device__ __forceinline__ WallRows wall_rows(const WallGeo &geo, bool back, int x) {
    const int first = back ? 3 : 0, next = back ? -1 : 1;
    const ColumnLine l0 = geo.line[first], l1 = geo.line[first + next], l2 = geo.line[first + 2 * next], l3 = geo.line[first + 3 * next];
    const HeightBend b0 = geo.bend[first], b1 = geo.bend[first + next], b2 = geo.bend[first + 2 * next], b3 = geo.bend[first + 3 * next];
    const int span0 = geo.span0, span1 = geo.span1;
    WallRows r;
    r.ceiling = height_row(l0, x); r.floor = height_row(l1, x);
    r.other_floor = height_row(l2, x); r.other_ceiling = height_row(l3, x);
    // nearly always every height of the linedef is one line over the whole screen
    if (__any((int)((b0.bottom | b1.bottom | b2.bottom | b3.bottom) >> 31))) {
        r.ceiling = bent_row(r.ceiling, b0, x); r.floor = bent_row(r.floor, b1, x);
        r.other_floor = bent_row(r.other_floor, b2, x); r.other_ceiling = bent_row(r.other_ceiling, b3, x);
    }
    if ((x < span0 || x >= span1) && ((b0.bottom | b1.bottom | b2.bottom | b3.bottom) >> 31)) {
        if (bends(b0)) r.ceiling = height_row(geo.outside[first], x);
        if (bends(b1)) r.floor = height_row(geo.outside[first + next], x);
        if (bends(b2)) r.other_floor = height_row(geo.outside[first + 2 * next], x);
        if (bends(b3)) r.other_ceiling = height_row(geo.outside[first + 3 * next], x);
    }
    return r;
}

// engine.py:10672-10739 (PrepWall) and 12762-12807: texture column before wrapping, texture step
template <typename Ends>
__device__ __forceinline__ void texture_column(const Ends &ends, bool past_left, const WallSide &ws, int side, int x, i64 *u_base, i64 *swall) {
    i64 h;
    texture_mapping(ends, ws.repeat, x, &h, swall);
    if (side != 0) h = ws.repeat - h;
    if (past_left && h < 0) h = 0;
    if (h >= ws.repeat) h = ws.repeat - 1;
    *u_base = (h + ws.offset_x) >> 16;
}

struct WallEnds { int tx0, tx1, ty0, ty1; };
// Exchanges inside the aligned groups of four lanes (DPP quads): the value of the group's first lane, and the
// conjunction, the largest and the smallest of the four.  All four lanes must be executing.
template <int PATTERN> __device__ __forceinline__ int quad_move(int v) { return __builtin_amdgcn_mov_dpp(v, PATTERN, 0xF, 0xF, true); }
__device__ __forceinline__ int quad_first(int v) { return quad_move<0x00>(v); }                 // lanes 0,0,0,0
__device__ __forceinline__ int quad_and(int v) { v &= quad_move<0xB1>(v); return v & quad_move<0x4E>(v); }   // lanes 1,0,3,2 then 2,3,0,1
__device__ __forceinline__ float quad_max(float v) {
    v = fmaxf(v, __int_as_float(quad_move<0xB1>(__float_as_int(v))));
    return fmaxf(v, __int_as_float(quad_move<0x4E>(__float_as_int(v))));
}
__device__ __forceinline__ float quad_min(float v) {
    v = fminf(v, __int_as_float(quad_move<0xB1>(__float_as_int(v))));
    return fminf(v, __int_as_float(quad_move<0x4E>(__float_as_int(v))));
}

// What one column draws of the drawseg a pass selected, as far as it depends on the selection alone and not on the column's clips
// (engine.py:12240-12807, 12969-13010).  A column's lanes prepare as many passes at once, one each, and pass them around (wall_raster_kernel).
// Of the up to two tiers of a drawseg, `a` is a one-sided drawseg's only one, or the lower one; `b` is the upper one.
struct PassDraw {
    unsigned int flags;       // DRAW_*; DRAW_SHADES: the column's own colormap row, then its group's; DRAW_BITS: floor(log2 height) of the tiers' textures
    unsigned int wall_sector; // the linedef | the sector drawn from << 16 | DRAW_MASKED
    unsigned int rows;        // the four heights' projected rows, not yet clipped: top, bottom, lower tier's top, upper tier's bottom
    unsigned int column_a, frac_a, step_a, column_b, frac_b, step_b;   // a tier's texture column in the atlas, its texture row (in the upper bits) at screen row 0, the step from row to row
    float distance;
};
#define DRAW_RASTER 0x1
#define DRAW_ONE_SIDED 0x2
#define DRAW_PS_KEEPS 0x4
#define DRAW_MARK_CEILING 0x8
#define DRAW_MARK_FLOOR 0x10
#define DRAW_LOWER 0x20       // the sector behind has the higher floor, or the lower ceiling
#define DRAW_UPPER 0x40
#define DRAW_TEXTURE_A 0x80
#define DRAW_TEXTURE_B 0x100
#define DRAW_CLIPS_BOTTOM 0x200   // the drawseg leaves a silhouette for the sprites behind it
#define DRAW_CLIPS_TOP 0x400
#define DRAW_GROUP 0x800      // the column's group of four draws this side of this linedef
#define DRAW_SHADES 12        // five bits each from here on
#define DRAW_BITS 22
#define DRAW_MASKED 0x20000000u   // a two-sided drawseg with a masked mid-texture (a sector's number has 13 bits: META_SECTOR_MASK)
static_assert(META_SECTOR_MASK < 1u << 13, "PassDraw packs a flag above the sector");

// A tier's texture row at screen row y is bits 32-height_bits .. 31 of
//   fraction(y) = (texture_mid << (16 - height_bits)) + ((step * (y * 65536 + 65536 - center)) >> 16).
// step * y * 65536 has no low 16 bits, so it shifts out of the floor unchanged, and only the low 32 bits of
// the sum are looked at: they advance by the low 32 bits of step per row, whatever the 64-bit terms wrap to.
__device__ __forceinline__ void tier_texture(const ColumnCtx &cc, int id, float origin, float offset_y, i64 u_base, i64 swall, unsigned &column, unsigned &frac, unsigned &step, unsigned &bits) {
    const Tables &tb = *cc.tb;
    bits = (unsigned)tb.height_bits(id);
    const i64 step64 = mul64(swall, shl64(1, 14 - (int)bits));
    const i64 base = shl64(round_to_i64((origin - cc.c->view_z) * 65536.0f + offset_y * 65536.0f), 16 - (int)bits);
    step = (unsigned)step64;
    frac = (unsigned)base + mul64_bits_16_47(step64, FIXED_UNIT - cc.c->center_fixed);
    column = (unsigned)id * (unsigned)(cc.m->tex_max_h * cc.m->tex_max_w) + (unsigned)tb.wrap_column(id, u_base);   // the atlas is below 4 GiB
}

// All of it is read off the lines wall_geometry_kernel left for the linedef (a pass marked REC_OWN_ROWS has its rows in
// Scratch::pass_rows); `at` is the record's place in the chunk's planes.  `draws`: the pass draws something; a column without a pass, or one whose pass
// draws nothing, paints no row and draws no tier.  The whole wavefront comes here.
template <bool GENERAL>
__device__ __forceinline__ PassDraw pass_draw(const DeviceMap &dm, const ColumnCtx &cc, const Scratch &sc, bool draws, const PassRec &rec, unsigned int geo_at, size_t at) {
    PassDraw d = {};
    const int x = cc.x;
    const int side = draws && (rec.marks & REC_SIDE1) ? 1 : 0, wi = draws ? (int)rec.wall : 0;
    const Tables &tb = *cc.tb;
    float light = 0.0f;
    i64 visibility = 0;
    if (draws) {
        const WallGeo &geo = sc.geo[geo_at];
        const WallSide ws = dm.wall_side[2 * wi + side];
        WallEnds ends;
        ends.tx0 = geo.tx0; ends.tx1 = geo.tx1; ends.ty0 = geo.ty0; ends.ty1 = geo.ty1;
        const bool past_left = geo.past_left != 0;
        const ColumnLine visibility_line = geo.visibility[side];
        const WallRows rows = wall_rows(geo, side != 0, x);
        visibility = visibility_line.at(x);
        if (GENERAL) {   // wallscan light interpolates over the fragment where a linedef has several
            const WallRec &wr = cc.rec(wi);
            const FragmentChoice fragment = choose_fragment<true>(cc.m, cc.frags, wr, wi, x);
            if (fragment.lights) visibility = wall_visibility(*fragment.rec, side, x);
        }
        // the sector behind only matters across a two-sided linedef (every use of its heights is behind !one_sided)
        d.rows = (unsigned)rows.ceiling | ((unsigned)rows.floor << 8) | ((unsigned)rows.other_floor << 16) | ((unsigned)rows.other_ceiling << 24);
        if (rec.marks & REC_OWN_ROWS) d.rows = sc.pass_rows[at].x;
        d.distance = rec.distance;
        const int current = rec.render_current, other = ws.other < 0 ? 0 : ws.other;
        const bool raster = rec.bits & PB_RASTER, one_sided = rec.bits & PB_ONE_SIDED, masked = !one_sided && ws.tex[0] >= 0;
        const float view_floor = tb.floor_h(current), view_ceiling = tb.ceil_h(current), other_floor = tb.floor_h(other), other_ceiling = tb.ceil_h(other);
        const float view_z = cc.c->view_z;
        light = (tb.light(current) + (float)(cc.c->flash_light * 16)) + ws.contrast;
        // k. plane marks (engine.py:12621-12636)
        const bool light_differs = tb.light(current) != tb.light(other);
        const bool mark_ceiling = one_sided || (view_ceiling != other_ceiling) || (tb.ceil_tex(current) != tb.ceil_tex(other)) || light_differs;
        const bool mark_floor = one_sided || (view_floor != other_floor) || (tb.floor_tex(current) != tb.floor_tex(other)) || light_differs;
        const bool lower = !one_sided && view_floor < other_floor, upper = !one_sided && view_ceiling > other_ceiling;
        const int tex_a = ws.tex[one_sided ? 0 : 1], tex_b = one_sided ? -1 : ws.tex[2];
        d.wall_sector = (unsigned)wi | ((unsigned)current << 16) | (masked ? DRAW_MASKED : 0u);
        d.flags = (raster ? DRAW_RASTER : 0) | (one_sided ? DRAW_ONE_SIDED : 0) | ((rec.bits & PB_PS_KEEPS) ? DRAW_PS_KEEPS : 0) | (mark_ceiling ? DRAW_MARK_CEILING : 0) |
                  (mark_floor ? DRAW_MARK_FLOOR : 0) | (lower ? DRAW_LOWER : 0) | (upper ? DRAW_UPPER : 0) | (tex_a >= 0 ? DRAW_TEXTURE_A : 0) | (tex_b >= 0 ? DRAW_TEXTURE_B : 0) |
                  // sprite silhouettes (engine.py:12943-12964)
                  (!one_sided && (view_floor > other_floor || view_z < other_floor || masked) ? DRAW_CLIPS_BOTTOM : 0) |
                  (!one_sided && (view_ceiling < other_ceiling || view_z > other_ceiling || masked) ? DRAW_CLIPS_TOP : 0);
        const bool paints_a = raster && tex_a >= 0 && (one_sided || lower), paints_b = raster && tex_b >= 0 && upper;
        if (paints_a || paints_b) {
            i64 u_base, swall;
            texture_column(ends, past_left, ws, side, x, &u_base, &swall);
            unsigned bits_a = 0, bits_b = 0;
            if (paints_a) tier_texture(cc, tex_a, one_sided ? view_ceiling : other_floor, ws.offset_y, u_base, swall, d.column_a, d.frac_a, d.step_a, bits_a);
            if (paints_b) tier_texture(cc, tex_b, other_ceiling, ws.offset_y, u_base, swall, d.column_b, d.frac_b, d.step_b, bits_b);
            d.flags |= (bits_a | (bits_b << 5)) << DRAW_BITS;
        }
    }
    // 4-column wallscan groups (engine.py:12688-12761): the four lanes of a group are one DPP quad, so every exchange is a vector move with
    // a lane pattern (no trip through the LDS crossbar).  Every lane of the wavefront is active here.
    const int wall_first = quad_first(wi), side_first = quad_first(side);
    const bool agrees = quad_and(wi == wall_first && side == side_first ? 1 : 0) != 0;
    const i64 group_visibility = ((i64)quad_first((int)(visibility >> 32)) << 32) | (i64)(unsigned)quad_first((int)(visibility & 0xFFFFFFFFLL));
    d.flags |= (agrees ? DRAW_GROUP : 0) | ((unsigned)wall_shade(light, visibility) << DRAW_SHADES) | ((unsigned)wall_shade(light, group_visibility) << (DRAW_SHADES + 5));
    return d;
}

// The rows of the portal path behind a projected solid (PB_PS_KEEPS, one pass in a thousand).
__device__ __forceinline__ WallRows path_rows(const ColumnCtx &cc, const Scratch &sc, size_t at, const PassRec &rec) {
    if (!(rec.marks & REC_OWN_ROWS)) return wall_rows(sc.geo[sc.geo_slot[cc.rec_base + (unsigned)rec.ps_path]], !(rec.bits & PB_PS_FROM_FRONT), cc.x);
    const unsigned int own = sc.pass_rows[at].y;
    WallRows rows;
    rows.ceiling = (float)(own & 255u); rows.floor = (float)((own >> 8) & 255u);
    rows.other_floor = (float)((own >> 16) & 255u); rows.other_ceiling = (float)(own >> 24);
    return rows;
}

// engine.py:12607-12620: the projected rows of a pass against the column's clips
struct PassRows { float top, bottom, upper_bottom, lower_top; };
__device__ __forceinline__ PassRows clip_pass(const PassDraw &d, float ceiling_clip, float floor_clip) {
    PassRows r;
    r.top = fmaxf((float)(d.rows & 255u), ceiling_clip);
    r.bottom = fminf((float)((d.rows >> 8) & 255u), floor_clip);
    r.upper_bottom = fmaxf(fminf((float)(d.rows >> 24), floor_clip), r.top);
    r.lower_top = fminf(fmaxf((float)((d.rows >> 16) & 255u), ceiling_clip), r.bottom);
    return r;
}

// engine.py:11769-12239: selection of the pass's drawseg for one column
template <bool SPLIT, int LANES>
__device__ __forceinline__ void pass_select(const ColumnCtx &cc, ListShare<LANES> &list, const ColumnState &c, bool boundary_has_po, PassColumn &r) {
    const gd_map_desc *m = cc.m;
    const MapView &mv = cc.mv;
    const int x = cc.x;
    const int cs = c.current_sector;
    const int cur = cs < 0 ? 0 : cs;
    const float prev = c.previous_distance;
    const float prev_eps = prev + 1e-3f;
    auto incident_c = [&](const ListEntry &q) { return MapView::incident(q.sectors, cur); };
    auto vertices_of = [&](const ListEntry &q) { return LANES > 1 ? q.vertices : mv.walls[q.wall].vertices; };
    // a. nearest incident linedef beyond previous_distance (engine.py:11769-11780)
    float distance = GD_INF; int wi = 0x7fffffff;
    Eval cwi;
    if constexpr (LANES == 1) list.begin(cc, prev);
    if (cs >= 0) {
        // b. equal-depth solid (engine.py:11784-11807): the nearest one-sided candidate replaces
        // the selection when it lies within 1e-3 of the nearest candidate, found in the same scan.
        u64 nearest = CAND_KEY_NONE, nearest_solid = CAND_KEY_NONE;
        auto take = [&](const ListEntry &q, bool there) {
            const u64 key = there && incident_c(q) && q.dist > prev ? q.key() : CAND_KEY_NONE;
            nearest = key < nearest ? key : nearest;
            const u64 solid_key = (q.flags & CF_ONE_SIDED) ? key : CAND_KEY_NONE;
            nearest_solid = solid_key < nearest_solid ? solid_key : nearest_solid;
        };
        if constexpr (LANES > 1) {
            list.each(cc, [&](const ListEntry &q) { take(q, true); });
            nearest = list.smallest(nearest); nearest_solid = list.smallest(nearest_solid);
        } else {
            list.template walk<true>(cc, take, [&]() { return cand_key_distance(nearest) + 2e-3f; });
        }
        const float sd = cand_key_distance(nearest_solid);
        if (finitef(sd) && (fabsf(sd - cand_key_distance(nearest)) <= 1e-3f)) nearest = nearest_solid;
        distance = cand_key_distance(nearest); wi = cand_key_wall(nearest);
        cwi.dist = distance; cwi.flags = cand_key_flags(nearest);
    }
    if (!finitef(distance)) { wi = 0; cwi = cc.first; }
    WallLinks links = mv.walls[wi];
    // c. selected endpoint (engine.py:11815-11871)
    bool sel_start = !(cwi.flags & CF_ALONG_HI);
    int sel_vertex = link_vertex(links.vertices, sel_start ? 0 : 1);
    auto shares_sel_c = [&](const ListEntry &q) { return MapView::has_vertex(vertices_of(q), sel_vertex); };
    bool continues_po_boundary = (c.flags & ST_PO) && (sel_vertex == c.pend_po_vertex);
    bool continues_ep_boundary = (c.flags & ST_EP) && (sel_vertex == c.pend_ep_vertex);
    int sel_slot = sel_start ? 0 : 1;
    // the forward bridge only matters while an endpoint-projected boundary continues
    int fb_idx = 0;
    bool pend_ep_has_forward_bridge = false;
    if (continues_ep_boundary && mv.portal_bridge(sel_slot, wi, links.sectors, links.vertices, c.pend_ep_wall, c.pend_ep_sectors, c.pend_ep_vertices, &fb_idx))
        pend_ep_has_forward_bridge = cc.eval(fb_idx).dist > distance + 1e-3f;
    bool completes_pending_endpoint_bridge = (c.flags & ST_EB) && (wi == c.pend_eb_index);
    bool sel_is_proj = cwi.flags & CF_PROJ;
    bool sel_excl_right = cwi.flags & CF_ENDS_HERE;
    // d. projected solid owner (engine.py:11872-11954)
    float ps_path_distance = distance; int ps_path_index = wi;
    const unsigned ps_sectors = links.sectors;
    bool ps_path_geo = cwi.flags & CF_GEO;
    float psd = GD_INF; int psi = 0x7fffffff; int psi_flags = 0;
    // A later scan of the pass, over all of a lane's own or, where a lane has the column alone, over `places` of the list.  `look` says whether `ask`, of which there is one copy, has to be asked about
    // the candidate as well.
    auto look_beyond = [&](u64 places, auto look, auto ask) {
        if constexpr (LANES > 1) {
            unsigned asked = 0;
#pragma unroll
            for (int j = 0; j < list.ENTRIES; ++j) asked |= look(list.own[j]) ? 1u << j : 0u;
            for (; asked; asked &= asked - 1) {
                ListEntry q = list.own[0];
#pragma unroll
                for (int j = 1; j < list.ENTRIES; ++j)
                    if ((asked & ((2u << j) - 1u)) == 1u << j) q = list.own[j];
                ask(q);
            }
        } else {
            list.each_of(cc, places, [&](const ListEntry &q) { if (look(q)) ask(q); });
        }
    };
    if (!sel_is_proj) {
        NearestOf<LANES> solid;
        u64 places = 0;
        if constexpr (LANES == 1) places = list.solid_ledges;
        look_beyond(places, [&](const ListEntry &q) {
            if (incident_c(q) && (q.flags & CF_ONE_SIDED) && (q.flags & CF_PROJ) && (q.flags & CF_LEDGE) && (q.dist > prev_eps) && shares_sel_c(q)) solid.take(q);
            return false;
        }, [](const ListEntry &) {});
        solid.share();
        psd = solid.distance(); psi = solid.wall(); psi_flags = solid.flags();
        if (sel_excl_right) {
            const int by_start = links.solid[0], by_end = links.solid[1];      // values: see WallLinks
            const int *idx = (sel_start ? m->solid_bridge_start_idx : m->solid_bridge_end_idx) + (sel_start ? by_start : by_end);
            const int bridges = sel_start ? links.solid_counts & 0xFFFFu : links.solid_counts >> 16;
            float sbd = GD_INF; int sbi = 0; int sbi_flags = 0;
            for (int k = 0; k < bridges; ++k) {
                int b = idx[k];
                const unsigned bridge_sectors = mv.walls[b].sectors;
                Eval q = cc.eval(b);
                if (!(MapView::incident(bridge_sectors, cur) && link_sector(bridge_sectors, 1) < 0)) continue;
                bool owner = (q.flags & CF_PROJ) && (q.flags & CF_LEDGE) && (q.dist > prev_eps);
                float v = owner ? q.dist : GD_INF;
                if (v < sbd) { sbd = v; sbi = b; sbi_flags = q.flags; }   // list is ascending: first slot wins ties
            }
            if (sbd < psd) { psd = sbd; psi = sbi; psi_flags = sbi_flags; }
        }
    }
    bool has_ps = finitef(psd);
    if (has_ps) { distance = psd; wi = psi; cwi.dist = psd; cwi.flags = psi_flags; links = mv.walls[wi]; }
    // e. endpoint owner (engine.py:11960-12001)
    int eo_idx; Eval eo;
    endpoint_owner(cc, wi, cwi, links, &eo_idx, &eo);
    bool eo_path_geo = cwi.flags & CF_GEO;
    bool replace_eo = (eo_idx != wi) && (eo.dist > prev_eps);
    unsigned sectors = links.sectors, vertices = links.vertices;     // wi's
    if (replace_eo) { distance = eo.dist; wi = eo_idx; cwi = eo; sectors = mv.walls[wi].sectors; vertices = mv.walls[wi].vertices; }
    int no_path_index = wi; float no_path_distance = distance;
    const unsigned no_path_sectors = sectors;
    bool no_path_geo = replace_eo ? eo_path_geo : (bool)(cwi.flags & CF_GEO);
    bool no_from_front = cs == link_sector(no_path_sectors, 0);
    int no_path_other = link_sector(no_path_sectors, no_from_front ? 1 : 0);
    // f. near projected owner (engine.py:12002-12179)
    bool so_is_proj = cwi.flags & CF_PROJ;
    const bool so_excl_right = cwi.flags & CF_ENDS_HERE, so_narrow = cwi.flags & CF_NARROW, so_short = cwi.flags & CF_SHORT;
    float npd = GD_INF; int npi = 0x7fffffff; int npi_flags = 0;
    if (!so_is_proj) {
        NearestOf<LANES> near;
        auto pairs_up = [&](const ListEntry &q) { return MapView::same_pair(q.sectors, sectors) && (fabsf(q.dist - distance) <= tolerance_of(q.dist)); };
        auto eligible = [&](const ListEntry &q) { return incident_c(q) && !(q.flags & CF_ONE_SIDED) && (q.flags & CF_PROJ) && (q.dist > prev_eps); };
        // A lane alone looks for the linedefs of the same pair of sectors about `distance` (a distance that is not finite has none), and for the others, which all
        // begin at this column, among those that do.
        if constexpr (LANES == 1) {
            if (finitef(distance))
                list.template walk<false>(cc, [&](const ListEntry &q, bool there) { if (there && eligible(q) && pairs_up(q)) near.take(q); },
                                          [&]() { return fmaxf(distance * 1.0080f, distance + 4.0f) + 0.25f; });
        }
        u64 places = 0;
        if constexpr (LANES == 1) places = so_excl_right && (so_narrow || so_short) ? list.ledges : 0;
        if (LANES > 1 || places != 0)
            look_beyond(places, [&](const ListEntry &q) {
                if (!eligible(q)) return false;
                bool le = q.flags & CF_LEDGE;
                bool close = pairs_up(q) || (le && so_excl_right && (so_narrow || (so_short && shares_sel_c(q))) && (fabsf(q.dist - distance) <= tolerance_of(q.dist)));
                if (close) near.take(q);
                return !close && le && so_excl_right && so_narrow;
            }, [&](const ListEntry &q) {
                int bridge; unsigned bridge_sectors;
                if (mv.sector_bridge(link_vertex(vertices_of(q), (q.flags & CF_ALONG_HI) ? 1 : 0), q.wall, q.sectors, no_path_index, no_path_sectors, &bridge, &bridge_sectors)) near.take(q);
            });
        near.share();
        npd = near.distance(); npi = near.wall(); npi_flags = near.flags();
    }
    int pe_wall = c.pend_ep_wall;
    int pe_s0 = link_sector(c.pend_ep_sectors, 0), pe_s1 = link_sector(c.pend_ep_sectors, 1);
    bool pe_from_current = cs == pe_s0;
    bool pe_incident = pe_from_current || (cs == pe_s1);
    int pe_other = pe_from_current ? pe_s1 : pe_s0;
    bool use_psb = false; int psb_idx = 0;
    if ((c.flags & ST_EP) && pe_incident && (pe_other >= 0) && (no_path_other >= 0) && no_path_geo && !so_is_proj && so_excl_right &&
        (cc.rec(pe_wall).sr - cc.rec(pe_wall).sl <= 1)) {
        int pe_slot = (c.pend_ep_vertex == link_vertex(c.pend_ep_vertices, 1)) ? 1 : 0;
        unsigned psb_sectors;
        bool psb_exists = mv.sector_bridge(link_vertex(c.pend_ep_vertices, pe_slot), pe_wall, c.pend_ep_sectors, no_path_index, no_path_sectors, &psb_idx, &psb_sectors);
        if (psb_exists) {
            int b0 = link_sector(psb_sectors, 0), b1 = link_sector(psb_sectors, 1);
            bool matches = (b0 == pe_other && b1 == no_path_other) || (b1 == pe_other && b0 == no_path_other);
            Eval qb = cc.eval(psb_idx);
            float pe_tol = tolerance_of(cc.eval(pe_wall).dist);
            bool psb = matches && (qb.flags & CF_PROJ) && (qb.flags & CF_LEDGE) && (qb.dist > prev - pe_tol) && (qb.dist < no_path_distance);
            if (psb && qb.dist < npd) { use_psb = true; npd = qb.dist; npi = psb_idx; npi_flags = qb.flags; }
        }
    }
    bool replace_np = finitef(npd);
    if (replace_np) { distance = npd; wi = npi; cwi.dist = npd; cwi.flags = npi_flags; sectors = mv.walls[wi].sectors; vertices = mv.walls[wi].vertices; }
    bool final_proj = cwi.flags & CF_PROJ, final_geo = cwi.flags & CF_GEO;
    bool completes_poab = (c.flags & ST_EP) && final_proj && !final_geo && mv.opposing(pe_wall, c.pend_ep_sectors, c.pend_ep_vertices, wi, sectors, vertices);
    // g. validity (engine.py:12197-12239)
    bool valid = finitef(distance);
    bool excl_only = !so_is_proj && so_excl_right && !replace_np && so_narrow && !boundary_has_po;
    bool raster_valid = valid && !excl_only && !continues_po_boundary &&
                        !((pend_ep_has_forward_bridge || completes_pending_endpoint_bridge) && !sel_is_proj && sel_excl_right && !replace_np);
    bool geometric_intersection = replace_np ? no_path_geo : (replace_eo ? eo_path_geo : final_geo);
    bool no_keeps = replace_np && no_path_geo && (no_path_other >= 0);
    // h. sides (engine.py:12240-12292)
    int front = link_sector(sectors, 0), back = link_sector(sectors, 1);
    bool from_front = cs == front;
    int other_sector = from_front ? back : front;
    int render_current = use_psb ? pe_other : (completes_poab ? other_sector : cur);
    bool render_from_front = render_current == front;
    int render_other = render_from_front ? back : front;
    int side = render_from_front ? 0 : 1;
    bool ps_from_front = cs == link_sector(ps_sectors, 0);
    int ps_other = link_sector(ps_sectors, ps_from_front ? 1 : 0);
    bool ps_keeps = has_ps && ps_path_geo && (ps_other >= 0);
    bool one_sided = other_sector < 0;

    // Can the rows of the pass be read off its linedefs' lines (WallGeo)?  Not through BSP fragments, and only where the sector
    // drawn from is the one its side (and its portal path's side) faces.
    bool own_rows = render_current != (render_from_front ? front : back) || (!one_sided && back < 0) ||
                    (ps_keeps && render_current != (ps_from_front ? cs : link_sector(ps_sectors, 1)));
    if (SPLIT) own_rows = own_rows || m->wall_split_slot[wi] >= 0 || (ps_keeps && m->wall_split_slot[ps_path_index] >= 0);
    r.marks = (side ? REC_SIDE1 : 0) | (own_rows ? REC_OWN_ROWS : 0);
    r.wall = wi; r.side = side; r.render_current = render_current; r.other_sector = other_sector;
    r.distance = distance; r.sectors = sectors; r.vertices = vertices;
    r.ps_path_index = ps_path_index; r.ps_other = ps_other; r.no_path_other = no_path_other; r.sel_vertex = sel_vertex; r.fb_idx = fb_idx;
    r.ps_path_distance = ps_path_distance; r.no_path_distance = no_path_distance;
    r.bits = (valid ? PB_VALID : 0) | (raster_valid ? PB_RASTER : 0) | (one_sided ? PB_ONE_SIDED : 0) |
             (ps_keeps ? PB_PS_KEEPS : 0) | (no_keeps ? PB_NO_KEEPS : 0) | (geometric_intersection ? PB_GEOMETRIC : 0) |
             (replace_np ? PB_REPLACE_NP : 0) | (ps_from_front ? PB_PS_FROM_FRONT : 0) | (continues_po_boundary ? PB_CONTINUES_PO : 0) |
             (pend_ep_has_forward_bridge ? PB_FORWARD_BRIDGE : 0) | ((cwi.flags & CF_ALONG_HI) ? PB_FINAL_ALONG_HI : 0);
}

// The per-pixel planes of a chunk of lanes and one column's place in them.  The wavefronts of the traversal hold columns of
// several lanes, so the planes' base pointers are the same for all of them and each column keeps byte offsets: a chunk
// is at most 4096 lanes, which keeps every offset below 4 GiB.
//
// The runs of rows are stored through buffer descriptors (put): a column that has nothing to store in a row the wavefront walks stores
// beyond the descriptor's end, which the hardware drops.  With a branch around the store instead, the compiler no longer knows how
// many stores are under way, so that the next use of a loaded texel waits for all of them to reach memory: every row
// waited for the row before (wall_raster_kernel, 4096 lanes on the 4000-linedef map: 1.33 ms with the branches, 1.03 without).
#define BUFFER_WORDS 0x00027000   // descriptor word 3: 32-bit elements
#define BUFFER_NOWHERE 0x80000000u   // an offset beyond every plane: 4096 lanes are 1.1 GB
template <int LANES> struct PixelBuffers {
    unsigned int *meta;     // [L][208][320]
    float *scene_depth;     // [L][208][320] or null
    __amdgpu_buffer_rsrc_t words, depths;   // meta and scene_depth once more, as buffers: see put()
    __amdgpu_buffer_rsrc_t bytes;           // the frame [L][240][320] or, where there is none, masked_texel [L][208][320]
    unsigned word_column;   // byte offset of (lane, row 0, column) in the four-byte planes
    unsigned put_byte_column;  // and in `bytes`, `row_lane` rows further on
    // A column may have several lanes of its wavefront (wall_raster_kernel): all of them hold the same state, and of the rows of a run
    // the lane `row_lane` of them takes every row_lanes-th, from the run's `row_lane`-th on.
    static constexpr int row_lanes = LANES;
    // a lane's rows per step of a walk over them.  Sixteen lanes take 64 rows a step: a run of 128 is rare, and a step costs what it has room for (16 lanes on
    // the 320-linedef map with 2 x 64 rows 37.2 us, 64 rows 33.9; eight lanes of four rows and of eight take the same)
    static constexpr int ROWS = LANES >= 16 ? 4 : 8;
    int row_lane;
    unsigned put_column;    // word_column, `row_lane` rows further on
    __device__ __forceinline__ unsigned int &m(int y) const { return *reinterpret_cast<unsigned int *>(reinterpret_cast<char *>(meta) + (word_column + (unsigned)y * (SW * 4u))); }
    // into row y + row_lane; `y` is the same in the whole wavefront
    __device__ __forceinline__ void put(bool active, int y, unsigned int word) const { __builtin_amdgcn_raw_buffer_store_b32(word, words, active ? put_column : BUFFER_NOWHERE, y * (SW * 4), 0); }
    // and out of it: zero for a lane that does not ask
    __device__ __forceinline__ unsigned int get(bool active, int y) const { return __builtin_amdgcn_raw_buffer_load_b32(words, active ? put_column : BUFFER_NOWHERE, y * (SW * 4), 0); }
    __device__ __forceinline__ void put_depth(bool active, int y, float depth) const { __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(depth), depths, active ? put_column : BUFFER_NOWHERE, y * (SW * 4), 0); }
    __device__ __forceinline__ void put_byte(bool active, int y, unsigned char byte) const { __builtin_amdgcn_raw_buffer_store_b8(byte, bytes, active ? put_byte_column : BUFFER_NOWHERE, y * SW, 0); }
    __device__ __forceinline__ float &s(int y) const { return *reinterpret_cast<float *>(reinterpret_cast<char *>(scene_depth) + (word_column + (unsigned)y * (SW * 4u))); }
};

// Silhouette bookkeeping: every row >= bot_row holds a clip depth <= bot_depth, every row
// < top_row holds a clip depth <= top_depth.  Clip depths only ever decrease, so a silhouette
// at a depth not below the bound cannot change those rows and they need not be visited.
// No clip recorded so far is deeper than `deepest`.
struct SilhouetteBounds {
    int bot_row, top_row;
    float bot_depth, top_depth, deepest;
};

// The ray distance of a linedef at this column: what the sprite clip of a row whose word names the linedef is at.  (Every clip is
// recorded with the distance the ray test of that linedef gives at that column, eval_segment's, so the word need not carry it.)
__device__ __forceinline__ float clip_distance(const ColumnCtx &cc, int w) {
    const float4 wl = *reinterpret_cast<const float4 *>(cc.m->walls + 4 * w);
    const float segx = wl.z - wl.x, segy = wl.w - wl.y, offx = wl.x - cc.c->x, offy = wl.y - cc.c->y;
    return (offx * segy - offy * segx) / (cc.rx * segy - cc.ry * segx);
}

// Rows that a silhouette may still change: they take its linedef as their sprite clip where it is nearer than what they hold.  `behind`: no clip of the column
// is deeper, so that only rows without any change, and nobody has to be asked how far a clip is.
struct ClipRun {
    int first, last;
    float distance;
    int wall;
    bool behind;
};
// The whole wavefront walks the rows together, as it does when it paints them (pass_paint): a few rows at a time, loads first, so that the rows' memory
// latencies overlap and neighbouring columns ask for neighbouring words.  With a loop a column over rows of its own, which asked for the distance of every other
// clip it met, silhouettes and masked mid-textures (masked_midtexture walks likewise) made wall_raster_kernel take 1013 us for 4096 lanes on the 4000-linedef map,
// 980 now; 2048 lanes with depths 496, 475; 1024 on the 2000-linedef map 232, 224.  (Notes of the claims that a silhouette will reach, so that it
// writes them anew without reading: 981 and 238, for the registers and the walks they take.)
template <typename Pixels>
__device__ __forceinline__ void clip_rows(const ColumnCtx &cc, const Pixels &pb, const ClipRun &run) {
    constexpr int ROWS = Pixels::ROWS;
    const unsigned rows = (unsigned)max(run.last - run.first, 0);
    if (!__any(rows != 0)) return;
    const int step = pb.row_lanes, wave_last = wave_max(rows ? run.last : 0);
    const bool asks = __any(rows != 0 && !run.behind);
    unsigned int held_wall = 0;           // linedef + 1 of the row before and its distance: rows of one clip are neighbours
    float held = GD_INF;
    wave_fence();                         // the column's other lanes may have written these rows
    for (int y = wave_min(rows ? run.first : VH); y < wave_last; y += ROWS * step) {
        unsigned int meta[ROWS]; bool takes[ROWS];
#pragma unroll
        for (int j = 0; j < ROWS; ++j) {
            takes[j] = (unsigned)(y + j * step + pb.row_lane - run.first) < rows;
            meta[j] = pb.get(takes[j], y + j * step);
        }
        if (!asks) {
#pragma unroll
            for (int j = 0; j < ROWS; ++j) takes[j] = takes[j] && (meta[j] & META_WALL_MASK) == 0;
        } else {
#pragma unroll
            for (int j = 0; j < ROWS; ++j) {
                const unsigned int row_wall = meta[j] & META_WALL_MASK;
                if (row_wall != held_wall && !run.behind) { held_wall = row_wall; held = row_wall ? clip_distance(cc, (int)row_wall - 1) : GD_INF; }
                takes[j] = takes[j] && (row_wall == 0 || (!run.behind && run.distance < held));
            }
        }
#pragma unroll
        for (int j = 0; j < ROWS; ++j) pb.put(takes[j], y + j * step, (meta[j] & ~META_WALL_MASK) | (unsigned)(run.wall + 1));
    }
}

// The rows that a bottom silhouette from `floor_clip` on and a top one up to `ceiling_clip` may change.
// `done_from` / `done_to`: rows [done_from, done_to) already carry this silhouette (pass_paint wrote it with
// the rows the pass took out of a window nothing had touched); an empty range otherwise.
__device__ __forceinline__ ClipRun bottom_run(SilhouetteBounds &sb, float floor_clip, float distance, int wall, int done_from, int done_to) {
    int first = floor_clip <= 0.0f ? 0 : (floor_clip >= (float)VH ? VH : (int)floor_clip);   // clips hold integers
    int last = (distance >= sb.bot_depth) ? (sb.bot_row < VH ? sb.bot_row : VH) : VH;
    const ClipRun run = {(done_to > first && done_from <= first) ? done_to : first, last, distance, wall, distance >= sb.deepest};
    sb.bot_row = first < sb.bot_row ? first : sb.bot_row;
    sb.bot_depth = fmaxf(sb.bot_depth, distance);
    return run;
}
__device__ __forceinline__ ClipRun top_run(SilhouetteBounds &sb, float ceiling_clip, float distance, int wall, int done_from, int done_to) {
    int end = ceiling_clip <= 0.0f ? 0 : (ceiling_clip >= (float)VH ? VH : (int)ceiling_clip);
    int start = (distance >= sb.top_depth) ? (sb.top_row > 0 ? sb.top_row : 0) : 0;
    const ClipRun run = {start, (done_from < end && done_to >= end) ? done_from : end, distance, wall, distance >= sb.deepest};
    sb.top_row = end > sb.top_row ? end : sb.top_row;
    sb.top_depth = fmaxf(sb.top_depth, distance);
    return run;
}

// May pass_paint write a two-sided pass's sprite silhouettes along with the rows the pass takes out of an untouched
// window?  Only while its lower and upper tier do not overlap on screen.
__device__ __forceinline__ bool silhouette_folds(const PassDraw &d, const PassRows &r) {
    return (d.flags & (DRAW_LOWER | DRAW_UPPER)) != (DRAW_LOWER | DRAW_UPPER) || !(r.lower_top < r.upper_bottom);
}

// The meta plane is never cleared between frames.  Instead the traversal keeps every row of its column that lies
// outside the open window [ceiling_clip, floor_clip) written (with a claim, a tier, or an explicit zero), reads no row
// inside the window until a one-sided drawseg has painted all of it, and zeroes what is left of the window when the
// column ends.  Rows that received such a zero are the only ones that can end up without an owner: the column keeps
// their range and lists the ownerless ones as gap pixels for the flat pass.
struct GapRange {
    // Four row numbers (0..VH, VH < 256) in one register: the traversal holds them for the whole column.
    //   bits 0-7 lo, 8-15 hi: rows [lo, hi) hold every zero this column wrote
    //   bits 16-23 filled_lo, 24-31 filled_hi: rows [filled_lo, filled_hi) are known to hold wall tier pixels
    //   (the one-sided drawseg's own)
    unsigned int rows;
    __device__ __forceinline__ int lo() const { return (int)(rows & 255u); }
    __device__ __forceinline__ int hi() const { return (int)((rows >> 8) & 255u); }
    __device__ __forceinline__ int filled_lo() const { return (int)((rows >> 16) & 255u); }
    __device__ __forceinline__ int filled_hi() const { return (int)(rows >> 24); }
    __device__ __forceinline__ void reset() { rows = (unsigned)VH; }
    __device__ __forceinline__ void set_zeroed(int lo, int hi) { rows = (rows & 0xffff0000u) | (unsigned)lo | ((unsigned)hi << 8); }
    __device__ __forceinline__ void set_filled(int lo, int hi) { rows = (rows & 0x0000ffffu) | ((unsigned)lo << 16) | ((unsigned)hi << 24); }
};
static_assert(VH < 256, "GapRange packs row numbers into bytes");
template <typename Pixels>
__device__ __forceinline__ void zero_rows(Pixels &pb, GapRange &gaps, int x, int first, int last) {
    first = first < 0 ? 0 : first; last = last > VH ? VH : last;
    if (first >= last) return;
    for (int y = first + pb.row_lane; y < last; y += pb.row_lanes) pb.m(y) = 0u;
    gaps.set_zeroed(min(first, gaps.lo()), max(last, gaps.hi()));
}

// engine.py:12637-12884
// `window_dirty` says whether some pixel inside the open window [ceiling_clip, floor_clip) may
// already be filled, plane-owned or carry a sprite-clip depth.  A two-sided drawseg only writes
// rows that its own clip update then removes from the window, so the window stays untouched
// until a one-sided drawseg (which leaves the clips alone) has painted; until then painting
// needs no reads and visits only the rows it writes.
template <bool DEPTH, typename Pixels>
__device__ __forceinline__ void pass_paint(const ColumnCtx &cc, const ColumnState &c, const PassDraw &d, const PassRows &r, Pixels &pb,
                           const bool group_valid[3], const float group_bottom[3], const unsigned char *colormap, bool &window_dirty, GapRange &gaps) {
    // The whole wavefront comes here together, columns with nothing to draw as well: they take part in the walks over the rows.
    const bool active = (d.flags & DRAW_RASTER) != 0;
    constexpr int ROWS = Pixels::ROWS;
    const gd_map_desc *m = cc.m;
    const int x = cc.x, wi = (int)(d.wall_sector & 0xFFFFu);
    const unsigned sector = (d.wall_sector >> 16) & META_SECTOR_MASK;
    const bool one_sided = d.flags & DRAW_ONE_SIDED, texture_a = d.flags & DRAW_TEXTURE_A, texture_b = d.flags & DRAW_TEXTURE_B;
    const float ceiling_plane_bottom = fminf(r.top, c.floor_clip);
    const float floor_plane_top = fmaxf(r.bottom, c.ceiling_clip);
    const unsigned char *own_shades = colormap + ((d.flags >> DRAW_SHADES) & 31u) * 256, *group_shades = colormap + ((d.flags >> (DRAW_SHADES + 5)) & 31u) * 256;
    // every span of this pass lies inside the open window [ceiling_clip, floor_clip)
    int y0 = c.ceiling_clip <= 0.0f ? 0 : (int)c.ceiling_clip;
    int y1 = c.floor_clip >= (float)VH ? VH : (int)c.floor_clip;
    const bool lower_on = d.flags & DRAW_LOWER, upper_on = d.flags & DRAW_UPPER;
    // a one-row texture (no bits) must shift everything out of its row: two shifts
    const unsigned shift_a = 31u - ((d.flags >> DRAW_BITS) & 31u), shift_b = 31u - (d.flags >> (DRAW_BITS + 5));
    const unsigned atlas_w = (unsigned)m->tex_max_w;
    const bool fresh = active && !window_dirty;
    if (__any(fresh)) {
        // clips and projections hold integers in [0, 208]
        const unsigned claim = (sector + 1u) << META_SECTOR_SHIFT;
        // The sprite silhouettes of a two-sided drawseg (engine.py:12943-12964) give every row that this pass
        // takes out of the window the pass's own (distance, linedef) as sprite clip.  Those rows are untouched
        // so far, so what this pass writes there carries the clip along and pass_advance need not revisit them:
        // tier rows hold it anyway, plane rows get it with their claim, rows left bare get it alone.
        // (Not where the lower and the upper tier overlap, a closed door say: a row of both that the lower tier
        // leaves undrawn for want of a texture would be missed.  silhouette_folds() is asked here and there.)
        const bool folds = !one_sided && silhouette_folds(d, r);
        const bool sil_bottom = folds && (d.flags & DRAW_CLIPS_BOTTOM), sil_top = folds && (d.flags & DRAW_CLIPS_TOP);
        const unsigned clip_word = (unsigned)(wi + 1);
        int ceiling_rows_end = 0; bool ceiling_claims = false;
        auto walk = [&](int first, int last, unsigned int word) {
            const unsigned rows = (unsigned)max(last - first, 0);
            for (int y = wave_min(first), wave_last = wave_max(last); y < wave_last; y += pb.row_lanes) pb.put((unsigned)(y + pb.row_lane - first) < rows, y, word);
        };
        {
            const bool claims = d.flags & DRAW_MARK_CEILING;
            const bool bare = !claims && sil_top && upper_on && texture_b;   // the upper tier lowers the clip past these rows
            // The wavefront walks the rows together, each column writing where its own range has the row: neighbouring
            // columns then store to neighbouring words, where loops that start at each column's own first row would
            // scatter every store over as many rows as the edges' slopes spread them.
            const bool writes = fresh && (claims || bare);
            const int first = writes ? (y0 < 0 ? 0 : y0) : VH, last = writes ? min((int)ceiling_plane_bottom, VH) : 0;
            const unsigned word = (claims ? claim : 0u) | (sil_top ? clip_word : 0u);
            walk(first, last, word);
            ceiling_rows_end = last; ceiling_claims = claims;
        }
        {
            const bool claims = d.flags & DRAW_MARK_FLOOR;
            const bool bare = !claims && sil_bottom && lower_on && texture_a;   // the lower tier raises the clip past these rows
            const bool writes = fresh && (claims || bare);
            const int first = writes ? max((int)floor_plane_top, 0) : VH, last = writes ? y1 : 0;
            const unsigned word = (claims ? (claim | META_FLOOR) : 0u) | (sil_bottom ? clip_word : 0u);
            walk(first, last, word);
            // A sector whose ceiling lies below its floor: the rows from its floor's row down to its ceiling's row
            // belong to both runs.  There the floor's claim has the say, the ceiling's stands where the floor makes none,
            // and the clip is recorded if either silhouette asks for it.
            if (__any(first < ceiling_rows_end)) {
                const int both_end = min(last, ceiling_rows_end);
                const unsigned both = (claims ? (claim | META_FLOOR) : (ceiling_claims ? claim : 0u)) | ((sil_top || sil_bottom) ? clip_word : 0u);
                for (int y = first + pb.row_lane; y < both_end; y += pb.row_lanes) pb.m(y) = both;
            }
        }
        // Rows that leave the window without being written: those the upper tier covers but that belong to a lower
        // tier without a texture (the lower tier has the say there), and a one-sided drawseg's own rows when it has none.
        if (fresh && lower_on && upper_on && !texture_a && texture_b)
            zero_rows(pb, gaps, x, max((int)r.top, (int)r.lower_top), min((int)r.upper_bottom, (int)r.bottom));
        if (fresh && one_sided && !texture_a) zero_rows(pb, gaps, x, max((int)r.top, y0), min((int)r.bottom, y1));
        int t0 = VH, t1 = 0;
        if (one_sided) { t0 = (int)r.top; t1 = (int)r.bottom; }
        if (lower_on) { t0 = min(t0, (int)r.lower_top); t1 = max(t1, (int)r.bottom); }
        if (upper_on) { t0 = min(t0, (int)r.top); t1 = max(t1, (int)r.upper_bottom); }
        const bool tiers_overlap = lower_on && upper_on && r.lower_top < r.upper_bottom;
        {
            // The usual case: the rows of a tier are one run, [top, bottom) of a one-sided drawseg, or the upper tier
            // above the lower one.  Each run is painted by a loop that knows its texture, so a row costs an add, a
            // shift, a texel, a colormap entry and the stores.  ROWS rows at a time, one batch ahead: the texels
            // of the next batch are asked for before the rows of this one are stored, so that a step waits for memory
            // once, not for its stores and then for its loads.
            // The wavefront walks the rows together (as above): neighbouring columns then read neighbouring texels and store
            // neighbouring words.  Each column starting at its own first row, every load and store touched 64 cache lines
            // (372 million cache accesses for 4096 lanes on the 4000-linedef map when a sprite clip plane was kept as well, 288 million now).
            // First run: a one-sided drawseg's rows, or the upper tier; second run: the lower tier.
            const bool runs = fresh && !tiers_overlap;
#pragma unroll 1
            for (int run = 0; run < 2; ++run) {   // one copy of the loop: the kernel is larger than the instruction cache as it is
                const bool second = run != 0;
                const bool tier_a = second || one_sided;
                int first = (int)(second ? r.lower_top : r.top), last = (int)(tier_a ? r.bottom : r.upper_bottom);
                const bool paints = runs && (second ? lower_on : one_sided || upper_on) && (tier_a ? texture_a : texture_b) && first < last;
                if (!__any(paints)) continue;
                first = paints ? first : VH; last = paints ? last : 0;
                const bool has_tail = second ? group_valid[1] : (one_sided ? group_valid[0] : group_valid[2]);
                const float tail_from = second ? group_bottom[1] : (one_sided ? group_bottom[0] : group_bottom[2]);
                const unsigned shift = tier_a ? shift_a : shift_b, step = tier_a ? d.step_a : d.step_b;
                const int wave_first = wave_min(first), wave_last = wave_max(last);
                const int stride = pb.row_lanes;
                unsigned frac = (tier_a ? d.frac_a : d.frac_b) + step * (unsigned)(wave_first + pb.row_lane);
                const unsigned advance = step * (unsigned)stride;
                // every texel asked for is the texture's own, whatever the row: the loads need no branch either.  (Of a tier that is not
                // there: the first texel of the atlas.)
                const unsigned column = tier_a ? d.column_a : d.column_b;
                // rows from tail_row on take the group's shade: (float)y >= tail_from, which no row meets if that is not a number
                const int tail_row = !has_tail || !(tail_from < (float)VH) ? VH : (tail_from <= 0.0f ? 0 : (int)ceilf(tail_from));
                const unsigned meta_word = META_FILLED | (unsigned)(wi + 1), rows = (unsigned)max(last - first, 0);
                auto load_rows = [&](unsigned char (&texel)[ROWS]) {
#pragma unroll
                    for (int j = 0; j < ROWS; ++j) { texel[j] = m->tex_atlas[column + __umul24((frac >> shift) >> 1, atlas_w)]; frac += advance; }
                };
                unsigned char texel[ROWS];
                load_rows(texel);
                for (int yb = wave_first; yb < wave_last; yb += ROWS * stride) {
                    const int y = yb + pb.row_lane;
                    unsigned char next_texel[ROWS]; unsigned colour[ROWS];
                    load_rows(next_texel);
#pragma unroll
                    for (int j = 0; j < ROWS; ++j) colour[j] = (y + j * stride >= tail_row ? group_shades : own_shades)[texel[j]];
#pragma unroll
                    for (int j = 0; j < ROWS; ++j) {
                        const bool own = (unsigned)(y + j * stride - first) < rows;
                        if (DEPTH) pb.put_depth(own, yb + j * stride, d.distance);
                        pb.put(own, yb + j * stride, meta_word | (colour[j] << META_SECTOR_SHIFT));
                    }
#pragma unroll
                    for (int j = 0; j < ROWS; ++j) texel[j] = next_texel[j];
                }
            }
        }
        if (fresh && tiers_overlap) {
            // The lower and the upper tier share rows (a closed door, say): the lower tier has the say there, row by row.
            unsigned frac_a = d.frac_a + d.step_a * (unsigned)t0, frac_b = d.frac_b + d.step_b * (unsigned)t0;
            // ROWS rows at a time, one batch ahead: the texels of the next batch are asked for before the rows of
            // this one are stored, so that a step waits for memory once, not for its stores and then for its loads
            auto load_rows = [&](int yb, unsigned char (&texel)[ROWS], unsigned &draw, unsigned &tail) {
                draw = 0; tail = 0;
#pragma unroll
                for (int j = 0; j < ROWS; ++j) {
                    const int y = yb + j;
                    const float py = (float)y;
                    const bool lower_span = (py >= r.lower_top) && (py < r.bottom);
                    const bool upper_span = (py >= r.top) && (py < r.upper_bottom);
                    const bool draws = y < t1 && (lower_span ? texture_a : upper_span && texture_b);
                    if (draws) draw |= 1u << j;
                    // rows that both tiers cover take the group's shade if either tier's common bottom has been passed
                    if ((lower_span && group_valid[1] && py >= group_bottom[1]) || (upper_span && group_valid[2] && py >= group_bottom[2])) tail |= 1u << j;
                    texel[j] = 0;
                    if (draws) {
                        const unsigned tv = ((lower_span ? frac_a >> shift_a : frac_b >> shift_b) >> 1);
                        texel[j] = m->tex_atlas[(lower_span ? d.column_a : d.column_b) + __umul24(tv, atlas_w)];
                    }
                    frac_a += d.step_a; frac_b += d.step_b;
                }
            };
            unsigned char texel[ROWS]; unsigned draw = 0, tail = 0;
            if (t0 < t1) load_rows(t0, texel, draw, tail);
            for (int yb = t0; yb < t1; yb += ROWS) {
                unsigned char next_texel[ROWS]; unsigned next_draw = 0, next_tail = 0;
#pragma unroll
                for (int j = 0; j < ROWS; ++j) next_texel[j] = 0;
                if (yb + ROWS < t1) load_rows(yb + ROWS, next_texel, next_draw, next_tail);
#pragma unroll
                for (int j = 0; j < ROWS; ++j) {
                    if (!(draw & (1u << j))) continue;
                    const unsigned colour = ((tail & (1u << j)) ? group_shades : own_shades)[texel[j]];
                    if (DEPTH) pb.s(yb + j) = d.distance;
                    pb.m(yb + j) = META_FILLED | (colour << META_SECTOR_SHIFT) | (unsigned)(wi + 1);
                }
#pragma unroll
                for (int j = 0; j < ROWS; ++j) texel[j] = next_texel[j];
                draw = next_draw; tail = next_tail;
            }
        }
        if (fresh && one_sided) {
            window_dirty = true;
            if (texture_a && t0 < t1) gaps.set_filled(max(t0, 0), min(t1, VH));   // every row of [t0, t1) was drawn just now
        }
    }
    if (!active || fresh) return;
    // A one-sided drawseg has painted this window.  Every row of it has been written since (GapRange), so what a later pass
    // can still change is narrow: a tier pixel where no tier was drawn yet, which can only lie in this pass's own tier rows
    // and outside the rows that drawseg filled, and a plane claim on a row nobody owns, which can only be one of the rows
    // this column had to zero.  Only those rows are visited (usually none).  Few columns come here (one pass in 300 on the
    // 4000-linedef map) but every eighth wavefront pass has one, so the loop is kept plain and light on registers.
    int lo = VH, hi = 0;
    if (one_sided) { lo = (int)r.top; hi = (int)r.bottom; }
    if (lower_on) { lo = min(lo, (int)r.lower_top); hi = max(hi, (int)r.bottom); }
    if (upper_on) { lo = min(lo, (int)r.top); hi = max(hi, (int)r.upper_bottom); }
    if (gaps.lo() < gaps.hi()) { lo = min(lo, gaps.lo()); hi = max(hi, gaps.hi()); }
    lo = max(lo, y0); hi = min(hi, y1);
    const int filled_lo = gaps.filled_lo(), filled_hi = gaps.filled_hi();
    const bool tail0 = group_valid[0], tail1 = group_valid[1], tail2 = group_valid[2];
    const float tail_row0 = group_bottom[0], tail_row1 = group_bottom[1], tail_row2 = group_bottom[2];
    wave_fence();                         // the column's other lanes may have written these rows
    for (int y = lo + pb.row_lane; y < hi; y += pb.row_lanes) {
        if (y >= filled_lo && y < filled_hi) { y += (filled_hi - 1 - y) & -pb.row_lanes; continue; }   // tier pixels already: nothing to add
        const float py = (float)y;
        unsigned int meta = pb.m(y);
        bool ceiling_span = (d.flags & DRAW_MARK_CEILING) && (py >= c.ceiling_clip) && (py < ceiling_plane_bottom);
        bool floor_span = (d.flags & DRAW_MARK_FLOOR) && (py >= floor_plane_top) && (py < c.floor_clip);
        bool meta_dirty = false;
        if (!(meta & META_FILLED) && ((meta >> META_SECTOR_SHIFT) & META_SECTOR_MASK) == 0 && (ceiling_span || floor_span)) {
            meta |= ((sector + 1u) << META_SECTOR_SHIFT) | (floor_span ? META_FLOOR : 0);
            meta_dirty = true;
        }
        bool one_span = one_sided && (py >= r.top) && (py < r.bottom);
        bool lower_span = lower_on && (py >= r.lower_top) && (py < r.bottom);
        bool upper_span = upper_on && (py >= r.top) && (py < r.upper_bottom);
        if (one_span || lower_span || upper_span) {
            const bool tier_a = one_span || lower_span;
            if ((tier_a ? texture_a : texture_b) && !(meta & META_FILLED)) {
                bool bottom_tail = (one_span && tail0 && py >= tail_row0) ||
                                   (lower_span && tail1 && py >= tail_row1) ||
                                   (upper_span && tail2 && py >= tail_row2);
                const unsigned fraction = (tier_a ? d.frac_a : d.frac_b) + (tier_a ? d.step_a : d.step_b) * (unsigned)y;
                const unsigned tv = (fraction >> (tier_a ? shift_a : shift_b)) >> 1;
                unsigned char texel = m->tex_atlas[(tier_a ? d.column_a : d.column_b) + __umul24(tv, atlas_w)];
                const unsigned colour = (bottom_tail ? group_shades : own_shades)[texel];
                if (DEPTH) pb.s(y) = d.distance;
                const float held = (meta & META_WALL_MASK) ? clip_distance(cc, (int)(meta & META_WALL_MASK) - 1) : GD_INF;   // no clip recorded yet
                if (d.distance < held) { meta = (meta & ~META_WALL_MASK) | (unsigned)(wi + 1); }
                meta = (meta & ~(META_SECTOR_MASK << META_SECTOR_SHIFT)) | (colour << META_SECTOR_SHIFT) | META_FILLED;
                meta_dirty = true;
            }
        }
        if (meta_dirty) pb.m(y) = meta;
    }
}

// engine.py:12885-13069: what a pass does to its column's clips, its masked drawseg snapshot and its sprite silhouettes.  The whole wavefront comes here
// together, columns whose pass does nothing as well (clip_rows).
template <typename Pixels>
__device__ __forceinline__ void advance_clips(const ColumnCtx &cc, ColumnState &c, const PassDraw &d, const PassRows &r, Pixels &pb, SilhouetteBounds &sb, bool window_untouched, GapRange &gaps,
                              const Scratch &sc, size_t at) {   // the pass's place in the chunk's planes
    const gd_map_desc *m = cc.m;
    const LaneCtx &L = *cc.c;
    const ColumnState before = c;
    const int x = cc.x, wi = (int)(d.wall_sector & 0xFFFFu);
    const float distance = d.distance;
    auto row_of = [](float clip) { return clip <= 0.0f ? 0 : (clip >= (float)VH ? VH : (int)clip); };
    const ClipRun nowhere = {VH, 0, 0.0f, 0, true};
    ClipRun bottom = nowhere, top = nowhere;
    if ((d.flags & (DRAW_RASTER | DRAW_ONE_SIDED)) == DRAW_RASTER) {
        // o. clip updates (engine.py:12888-12913)
        const bool draws_upper = (d.flags & (DRAW_UPPER | DRAW_TEXTURE_B)) == (DRAW_UPPER | DRAW_TEXTURE_B), draws_lower = (d.flags & (DRAW_LOWER | DRAW_TEXTURE_A)) == (DRAW_LOWER | DRAW_TEXTURE_A);
        if (draws_upper || (d.flags & DRAW_MARK_CEILING)) c.ceiling_clip = draws_upper ? r.upper_bottom : r.top;
        if (draws_lower || (d.flags & DRAW_MARK_FLOOR)) c.floor_clip = draws_lower ? r.lower_top : r.bottom;
        // p. masked drawseg snapshot (engine.py:12914-12939)
        if ((d.wall_sector & DRAW_MASKED) && distance < c.masked_distance) {
            c.masked_ceiling_clip = c.ceiling_clip; c.masked_floor_clip = c.floor_clip; c.masked_distance = distance; c.masked_wall = wi;
        }
        // q. sprite silhouettes (engine.py:12943-12964)
        const bool bottom_sil = d.flags & DRAW_CLIPS_BOTTOM, top_sil = d.flags & DRAW_CLIPS_TOP;
        // pass_paint, finding the window untouched, has written the silhouette into the rows that this pass took out
        // of it: [new floor clip, old floor clip) at the bottom, [old ceiling clip, new ceiling clip) at the top
        const int old_floor = row_of(before.floor_clip), old_ceiling = row_of(before.ceiling_clip);
        // (pass_paint stays inside the old window, and a sector whose ceiling lies below its floor can carry a clip past the window's other end: then the
        // rows beyond that end are not done, and the range is cut there: all of them are visited.)
        const bool folded = window_untouched && silhouette_folds(d, r);
        if (bottom_sil) bottom = bottom_run(sb, c.floor_clip, distance, wi, folded ? max(row_of(c.floor_clip), old_ceiling) : 0, folded ? old_floor : 0);
        if (top_sil) top = top_run(sb, c.ceiling_clip, distance, wi, folded ? old_ceiling : 0, folded ? min(row_of(c.ceiling_clip), old_floor) : 0);
    }
    clip_rows(cc, pb, bottom);
    clip_rows(cc, pb, top);
    if (d.flags & DRAW_RASTER) sb.deepest = fmaxf(sb.deepest, distance);     // what the pass painted shows its linedef
    if (!__any(d.flags & DRAW_PS_KEEPS)) return;
    // r. clips of the geometric portal behind a projected solid (engine.py:12969-13069)
    bottom = nowhere; top = nowhere;
    if (d.flags & DRAW_PS_KEEPS) {
        const PassRec rec = sc.pass_rec[at];
        const int path = rec.ps_path, current = rec.render_current;
        const int path_safe_other = rec.ps_other < 0 ? 0 : rec.ps_other;
        const Tables &tb = *cc.tb;
        const float view_floor = tb.floor_h(current), view_ceiling = tb.ceil_h(current);
        float pof = tb.floor_h(path_safe_other), poc = tb.ceil_h(path_safe_other);
        int pside = (rec.bits & PB_PS_FROM_FRONT) ? 0 : 1;
        const int *ptex = m->side_tex + (path * 2 + pside) * 3;
        const WallRows rows = path_rows(cc, sc, at, rec);
        const float path_distance = sc.pass_path_distance[at];
        float pct = fmaxf(rows.ceiling, c.ceiling_clip);
        float pcb = fminf(rows.floor, c.floor_clip);
        float pcub = fmaxf(fminf(rows.other_ceiling, c.floor_clip), pct);
        float pclt = fminf(fmaxf(rows.other_floor, c.ceiling_clip), pcb);
        bool light_differs = tb.light(current) != tb.light(path_safe_other);
        bool p_draws_upper = (view_ceiling > poc) && (ptex[2] >= 0);
        bool p_marks_ceiling = (view_ceiling != poc) || (tb.ceil_tex(current) != tb.ceil_tex(path_safe_other)) || light_differs;
        bool p_draws_lower = (view_floor < pof) && (ptex[1] >= 0);
        bool p_marks_floor = (view_floor != pof) || (tb.floor_tex(current) != tb.floor_tex(path_safe_other)) || light_differs;
        float new_ceiling = c.ceiling_clip, new_floor = c.floor_clip;
        if (p_draws_upper || p_marks_ceiling) new_ceiling = p_draws_upper ? pcub : pct;
        if (p_draws_lower || p_marks_floor) new_floor = p_draws_lower ? pclt : pcb;
        if (window_untouched) {
            // These clips move without anything being painted or claimed: the rows they take out of an untouched
            // window would leave it unwritten.  They show the flat pass's picture.
            const int window_top = row_of(c.ceiling_clip), window_bottom = row_of(c.floor_clip);
            zero_rows(pb, gaps, x, window_top, min(row_of(new_ceiling), window_bottom));
            zero_rows(pb, gaps, x, max(row_of(new_floor), window_top), window_bottom);
        }
        c.ceiling_clip = new_ceiling; c.floor_clip = new_floor;
        bool pmasked = ptex[0] >= 0;
        bool pbottom = (view_floor > pof) || (L.view_z < pof) || pmasked;
        bool ptop = (view_ceiling < poc) || (L.view_z > poc) || pmasked;
        if (pbottom) bottom = bottom_run(sb, c.floor_clip, path_distance, path, 0, 0);
        if (ptop) top = top_run(sb, c.ceiling_clip, path_distance, path, 0, 0);
        sb.deepest = fmaxf(sb.deepest, path_distance);
    }
    clip_rows(cc, pb, bottom);
    clip_rows(cc, pb, top);
}

// engine.py:13070-13371: where a pass takes its column's traversal: next sector, previous distance, pending boundaries
template <bool SPLIT, int LANES>
__device__ __forceinline__ bool pass_advance(const ColumnCtx &cc, ListShare<LANES> &list, ColumnState &c, const PassColumn &r) {
    const gd_map_desc *m = cc.m;
    const MapView &mv = cc.mv;
    const LaneCtx &L = *cc.c;
    const ColumnState before = c;
    const int x = cc.x;
    const int cs = c.current_sector;
    const int cur = cs < 0 ? 0 : cs;
    const int wi = r.wall;
    const float distance = r.distance;
    const bool valid = r.bits & PB_VALID, one_sided = r.bits & PB_ONE_SIDED;
    // s. next sector (engine.py:13070-13241)
    const float prior = before.previous_distance;
    const float prior_eps = prior + 1e-3f;
    const bool geometric_intersection = r.bits & PB_GEOMETRIC;
    bool endpoint_only_portal = valid && !one_sided && !geometric_intersection;
    const int other_sector = r.other_sector;
    float pd = prior;
    int next_sector = -1;
    bool endpoint_portal_bridge = false;
    int ppb_idx = 0, gp_other = -1; float gpd = GD_INF;
    if (endpoint_only_portal) {
        const float dist_eps = distance + 1e-3f;
        NearestOf<LANES> current_next, other_next, geometric;
        const unsigned none = __float_as_uint(GD_INF);
        unsigned current_solid = none, other_solid = none;      // distances: positive, so their bits order as they do
        const int v0 = link_vertex(r.vertices, 0), v1 = link_vertex(r.vertices, 1);
        auto look = [&](const ListEntry &q, bool there) {
            const float d = q.dist;
            if (!there) return;
            bool os = q.flags & CF_ONE_SIDED;
            bool inc = MapView::incident(q.sectors, cur), oinc = MapView::incident(q.sectors, other_sector);
            bool future = ((q.flags & CF_GEO) || os) && (d > dist_eps);
            if (future && inc) current_next.take(q);
            if (future && oinc) other_next.take(q);
            bool shared_solid = os && (inc || oinc) && (d > prior_eps) && (d <= dist_eps);
            bool sgp = (q.flags & CF_GEO) && inc && !os && (d > prior_eps) && (fabsf(d - distance) <= (1.0f / 16.0f));
            if (sgp || (shared_solid && !(q.flags & CF_LEDGE))) {      // few of them: a lane alone asks memory for the vertices
                const unsigned vertices = LANES > 1 ? q.vertices : mv.walls[q.wall].vertices;
                const bool shares_endpoint = MapView::has_vertex(vertices, v0) || MapView::has_vertex(vertices, v1);
                sgp = sgp && shares_endpoint; shared_solid = shared_solid && shares_endpoint;
            }
            if (shared_solid && inc) current_solid = min(current_solid, __float_as_uint(d));
            if (shared_solid && oinc) other_solid = min(other_solid, __float_as_uint(d));
            if (sgp) geometric.take(q);
        };
        if constexpr (LANES > 1) list.each(cc, [&](const ListEntry &q) { look(q, true); });
        else {
            // Which of the two next ones is nearer is all that matters: with one of them found, what the other is beyond it does not.  (But for linedef 0 next
            // in the current sector, which a search for the other's that finds none counts as tied with.)
            list.template walk<false>(cc, look, [&]() {
                const float cnd = current_next.distance(), ond = other_next.distance();
                return fmaxf(cnd <= ond && current_next.wall() == 0 ? ond : fminf(cnd, ond), distance + 0.07f);
            });
        }
        current_next.share(); other_next.share(); geometric.share();
        current_solid = list.smallest(current_solid); other_solid = list.smallest(other_solid);
        const float cnd = current_next.distance(), ond = other_next.distance(), csd = __uint_as_float(current_solid), osd = __uint_as_float(other_solid);
        int cni = current_next.wall(), oni = other_next.wall();
        const int gpi = geometric.wall();
        const bool gp_along_hi = (geometric.flags() & CF_ALONG_HI) != 0;
        gpd = geometric.distance();
        if (!finitef(cnd)) cni = 0;
        if (!finitef(ond)) oni = 0;
        bool enters_tied_strip = false;
        if (finitef(cnd) && cni == oni) { const WallLinks &tied = mv.walls[cni]; enters_tied_strip = mv.opposing(wi, r.sectors, r.vertices, cni, tied.sectors, tied.vertices); }
        bool enters_other = (other_sector >= 0) && ((ond < cnd) || enters_tied_strip);
        bool enters_shared = (other_sector >= 0) && (osd < csd);
        bool uses_geometric_path = false;
        if (finitef(gpd)) {
            const unsigned gp_sectors = mv.walls[gpi].sectors, gp_vertices = mv.walls[gpi].vertices;
            bool gp_from_front = cs == link_sector(gp_sectors, 0);
            gp_other = link_sector(gp_sectors, gp_from_front ? 1 : 0);
            uses_geometric_path = gp_other >= 0;
            if (uses_geometric_path) {
                int pb_slot = gp_along_hi ? 1 : 0;
                bool ppb_exists = mv.portal_bridge(pb_slot, gpi, gp_sectors, gp_vertices, wi, r.sectors, r.vertices, &ppb_idx);
                if (ppb_exists) {
                    Eval qb = cc.eval(ppb_idx);
                    endpoint_portal_bridge = (qb.flags & CF_PROJ) && (qb.flags & CF_LEDGE) && (qb.dist > prior_eps) && (fabsf(qb.dist - gpd) <= tolerance_of(gpd));
                }
            }
        }
        // t. previous_distance (engine.py:13242-13262)
        if (r.bits & PB_NO_KEEPS) pd = r.no_path_distance;
        else if (r.bits & PB_PS_KEEPS) pd = r.ps_path_distance;
        else if (enters_shared && (osd < distance)) pd = prior;
        else if (uses_geometric_path) pd = gpd;
        else pd = distance;
        if (r.bits & PB_NO_KEEPS) next_sector = r.no_path_other;
        else if (r.bits & PB_PS_KEEPS) next_sector = r.ps_other;
        else if (uses_geometric_path) next_sector = gp_other;
        else if (enters_other || enters_shared) next_sector = other_sector;
        else next_sector = cs;
    } else {
        if (valid) {
            if (r.bits & PB_NO_KEEPS) pd = r.no_path_distance;
            else if (r.bits & PB_PS_KEEPS) pd = r.ps_path_distance;
            else pd = distance;
        }
        if (r.bits & PB_NO_KEEPS) next_sector = r.no_path_other;
        else if (r.bits & PB_PS_KEEPS) next_sector = r.ps_other;
        else if (valid && !one_sided && geometric_intersection) next_sector = other_sector;
        else next_sector = -1;
    }
    bool completes_pending_portal_bridge = valid && (before.flags & ST_PB) && (wi == before.pend_pb_index);
    if (valid && endpoint_portal_bridge) pd = prior;
    if (valid && completes_pending_portal_bridge) pd = fmaxf(distance, before.pend_pb_exit);
    c.previous_distance = pd;
    // carried state (engine.py:13276-13313, 13355-13371)
    bool starts_po = r.bits & PB_REPLACE_NP;
    if (starts_po) c.pend_po_vertex = r.sel_vertex;
    bool po = starts_po || ((before.flags & ST_PO) && (r.bits & PB_CONTINUES_PO));
    if (endpoint_only_portal) {
        c.pend_ep_vertex = link_vertex(r.vertices, (r.bits & PB_FINAL_ALONG_HI) ? 1 : 0);
        c.pend_ep_wall = wi; c.pend_ep_sectors = r.sectors; c.pend_ep_vertices = r.vertices;
    }
    if (r.bits & PB_FORWARD_BRIDGE) c.pend_eb_index = r.fb_idx;
    if (endpoint_portal_bridge) next_sector = other_sector;
    if (completes_pending_portal_bridge) next_sector = before.pend_pb_sector;
    if (endpoint_portal_bridge) { c.pend_pb_index = ppb_idx; c.pend_pb_sector = gp_other; c.pend_pb_exit = gpd; }
    c.flags = (po ? ST_PO : 0) | (endpoint_only_portal ? ST_EP : 0) | ((r.bits & PB_FORWARD_BRIDGE) ? ST_EB : 0) | (endpoint_portal_bridge ? ST_PB : 0);
    c.current_sector = next_sector;
    return !same_state(before, c);
}

// engine.py:13424-13744 for one column; the whole wavefront comes here
template <bool DEPTH, bool GENERAL, typename Pixels>
__device__ __forceinline__ void masked_midtexture(const DeviceMap &dm, const ColumnCtx &cc, const Scratch &sc, int local, const ColumnState &c, Pixels &pb, const unsigned char *colormap) {
    constexpr int ROWS = Pixels::ROWS;
    const gd_map_desc *m = cc.m;
    const LaneCtx &L = *cc.c;
    const int x = cc.x;
    const u64 hit = sc.masked_hit[(size_t)local * SW + x];
    const int mw = cand_key_wall(hit), cand_flags = cand_key_flags(hit);
    const float md = cand_key_distance(hit);
    const int mside = (cand_flags & CF_FF) ? 0 : 1;   // engine.py:13436-13444, the float32 facing test
    bool left_edge = cand_flags & CF_LEDGE;
    bool has_saved = c.masked_wall == mw;
    const bool shows = hit != CAND_KEY_NONE && (has_saved || left_edge);
    if (!__any(shows)) return;
    // what a column walks over its rows with: none of them, and the first texel of the atlas
    int y0 = VH, y1 = 0;
    unsigned row_step = 0, row_base = 0, texel_base = 0, shift = 0, shades = 0;
    if (shows) {
        const WallSide &ws = dm.wall_side[2 * mw + mside];
        const WallGeo &geo = sc.geo[sc.geo_slot[cc.rec_base + (unsigned)mw]];
        const MaskedGeo &masked = sc.masked_geo[(size_t)local * dm.masked_count + dm.masked_slot[mw]];
        const int texture_id = ws.tex[0];
        const Tables &tb = *cc.tb;
        const int front_sector = m->wall_sectors[2 * mw], back_sector = m->wall_sectors[2 * mw + 1];
        const int light_sector = mside == 0 ? front_sector : back_sector;
        const float world_top = fminf(tb.ceil_h(front_sector), tb.ceil_h(back_sector));
        const int th = m->tex_h[texture_id];   // the texture's own height, whatever its row mask (engine.py:13480-13483)
        float owall_top, owall_bottom;
        i64 visibility = geo.visibility[mside].at(x);
        bool split = false;
        if (GENERAL) {
            const WallRec &wr = cc.rec(mw);
            split = (wr.flags & WF_SPLIT) != 0;
            if (split) {
                const FragmentChoice fragment = choose_fragment<true>(m, cc.frags, wr, mw, x);
#pragma unroll 1
                for (int k = 0; k < 2; ++k) {
                    float v = project(L, wr, fragment, k == 0 ? world_top : world_top - (float)th, x);
                    if (k == 0) owall_top = v; else owall_bottom = v;
                }
                if (fragment.lights) visibility = wall_visibility(*fragment.rec, mside, x);
            }
        }
        if (!split) {
            const bool in_span = x >= geo.span0 && x < geo.span1;
            const HeightBend top_bend = masked.bend[0], bottom_bend = masked.bend[1];
            owall_top = !in_span && bends(top_bend) ? height_row(masked.outside[0], x) : bent_row(height_row(masked.line[0], x), top_bend, x);
            owall_bottom = !in_span && bends(bottom_bend) ? height_row(masked.outside[1], x) : bent_row(height_row(masked.line[1], x), bottom_bend, x);
        }
        float mceil = fmaxf(owall_top, has_saved ? c.masked_ceiling_clip : 0.0f);
        float mfloor = fminf(owall_bottom, has_saved ? c.masked_floor_clip : (float)VH);
        i64 u_base, swall_cur;
        texture_column(geo, geo.past_left != 0, ws, mside, x, &u_base, &swall_cur);
        const i64 mu = tb.wrap_column(texture_id, u_base);
        int height_bits = ilog2(th);
        i64 vertical_step = mul64(swall_cur, shl64(1, 14 - height_bits));
        i64 center_fixed = L.center_fixed;
        i64 texture_mid = round_to_i64((world_top - L.view_z) * 65536.0f + ws.offset_y * 65536.0f);
        const i64 sprite_scale = masked.scale.at(x);
        i64 top_screen = center_fixed - (mul64(texture_mid, sprite_scale) >> 16);
        i64 post_top = top_screen >> 16;
        i64 post_bottom = ((top_screen + mul64(sprite_scale, th) - FIXED_UNIT) >> 16) + 1;
        i64 clipped_top = max64(post_top, (i64)mceil);
        i64 clipped_bottom = min64(post_bottom, (i64)mfloor);
        i64 dc_iscale = mul64(swall_cur, FIXED_UNIT) >> 18;
        bool initial_post = clipped_top < clipped_bottom;
        i64 frac_start = texture_mid + mul64(clipped_top, dc_iscale) - (mul64(center_fixed - FIXED_UNIT, dc_iscale) >> 16);
        i64 frac_end = frac_start + mul64(clipped_bottom - clipped_top - 1, dc_iscale);
        bool extends = initial_post && ((float)clipped_bottom < mfloor) && (frac_end < (i64)th * FIXED_UNIT - dc_iscale);
        clipped_bottom += extends ? 1 : 0;
        float light = (tb.light(light_sector) + (float)(L.flash_light * 16)) + ws.contrast;
        shades = (unsigned)wall_shade(light, visibility) * 256u;
        y0 = (int)clampi(clipped_top, 0, VH); y1 = (int)clampi(clipped_bottom, 0, VH);
        // as in pass_paint: only the low 32 bits of the row fraction matter, and they advance by the step's low 32 bits
        row_step = (unsigned)vertical_step;
        row_base = (unsigned)(shl64(texture_mid, 16 - height_bits) + (mul64(vertical_step, FIXED_UNIT - center_fixed) >> 16));
        texel_base = (unsigned)texture_id * (unsigned)(m->tex_max_h * m->tex_max_w) + (unsigned)mu;    // the atlas is below 4 GiB
        shift = 31u - (unsigned)height_bits;
    }
    // The wavefront walks the rows together (pass_paint).  The texel goes to the frame where there is one; otherwise it waits for the kernel that assembles
    // the frame.
    const unsigned atlas_w = (unsigned)m->tex_max_w, rows = (unsigned)max(y1 - y0, 0);
    const int stride = pb.row_lanes, wave_last = wave_max(rows ? y1 : 0);
    wave_fence();                         // the column's other lanes may have written these rows
    for (int yb = wave_min(rows ? y0 : VH); yb < wave_last; yb += ROWS * stride) {
        unsigned char texel[ROWS]; unsigned int word[ROWS];
#pragma unroll
        for (int j = 0; j < ROWS; ++j) {
            const int y = yb + j * stride + pb.row_lane;
            texel[j] = m->tex_atlas[texel_base + __umul24(((row_base + row_step * (unsigned)y) >> shift) >> 1, atlas_w)];
            word[j] = pb.get((unsigned)(y - y0) < rows, yb + j * stride);
        }
#pragma unroll
        for (int j = 0; j < ROWS; ++j) {
            const bool own = (unsigned)(yb + j * stride + pb.row_lane - y0) < rows;
            pb.put_byte(own, yb + j * stride, colormap[shades + texel[j]]);
            pb.put(own, yb + j * stride, word[j] | META_MASKED);
            if (DEPTH) pb.put_depth(own, yb + j * stride, md);
        }
    }
}

// One height of a linedef as a line over the columns: OWallMost (engine.py:12294-12605, project() above) with the column left open.
struct HeightLine { ColumnLine line, outside; HeightBend bend; };
__device__ __forceinline__ HeightLine height_line(const LaneCtx &c, const WallRec &g, float world_z) {
    HeightLine out;
    const i64 depth_left = max64(g.dl, 1), depth_right = max64(g.dr, 1);
    const i64 pz = -(round_to_i64((world_z - c.view_z) * 65536.0f) >> 4);
    auto line_of = [&](i64 left, i64 right, i64 dl, i64 dr) {
        const i64 pl = tdiv(mul64(pz, FOCAL_Y_FIXED), max64(dl, 1)), pr = tdiv(mul64(pz, FOCAL_Y_FIXED), max64(dr, 1));
        ColumnLine line;
        line.step = tdiv(pr - pl, max64(right - left, 1));
        line.base = (i64)((u64)(c.center_fixed + pl) - (u64)left * (u64)line.step);
        return line;
    };
    out.outside = line_of(g.sl, g.sr, depth_left, depth_right);
    out.line = out.outside;
    out.bend.top = 0u; out.bend.bottom = 0u;
    if (!(g.sr > g.sl)) return out;
    const i64 upper_left = mul64(c.upper_clip, depth_left) >> 16, upper_right = mul64(c.upper_clip, depth_right) >> 16;
    const i64 lower_left = mul64(c.lower_clip, depth_left) >> 16, lower_right = mul64(c.lower_clip, depth_right) >> 16;
    const bool above_left = pz < upper_left, above_right = pz < upper_right;
    const bool below_left = pz > lower_left, below_right = pz > lower_right;
    const bool entirely_above = above_left && above_right, entirely_below = below_left && below_right;
    const bool crosses_top = above_left != above_right, crosses_bottom = below_left != below_right;
    if (!(entirely_above || entirely_below || crosses_top || crosses_bottom)) return out;
    out.bend.bottom = 0x80000000u;
    i64 clipped_left = g.sl, clipped_right = g.sr, clipped_dl = depth_left, clipped_dr = depth_right;
    i64 top0 = 0, top1 = 0, bottom0 = 0, bottom1 = 0;
#pragma unroll 1
    for (int edge = 0; edge < 2; ++edge) {   // the top of the view, then its bottom: one copy of the divisions
        if (!(edge ? crosses_bottom : crosses_top)) continue;
        const i64 at_left = edge ? lower_left : upper_left, at_right = edge ? lower_right : upper_right;
        const bool beyond_left = edge ? below_left : above_left, beyond_right = edge ? below_right : above_right;
        const i64 fraction = tdiv(shl64(pz - at_left, 30), at_right != at_left ? at_right - at_left : 1);
        const i64 depth = depth_left + (mul64(depth_right - depth_left, fraction) >> 30);
        const i64 cross = g.sl + tdiv(mul64(mul64(depth_right, fraction) >> 30, g.sr - g.sl), max64(depth, 1));
        if (beyond_right && g.sl <= cross) { clipped_right = cross; clipped_dr = depth; }
        if (beyond_left && cross <= g.sr) { clipped_left = cross; clipped_dl = depth; }
        const i64 from = beyond_right ? cross : g.sl, to = beyond_right ? g.sr : cross;   // the columns beyond the edge
        if (edge) { bottom0 = from; bottom1 = to; } else { top0 = from; top1 = to; }
    }
    auto column = [](i64 v) { return (unsigned int)clampi(v, 0, SW); };
    if (entirely_above) {
        out.line.base = 0; out.line.step = 0;
        return out;
    }
    out.bend.top = column(top0) | (column(top1) << 10);
    if (entirely_below) {
        out.line.base = (i64)VH << 16; out.line.step = 0;
        return out;
    }
    out.bend.bottom |= column(bottom0) | (column(bottom1) << 10);
    if (clipped_right == clipped_left && clipped_left >= 0 && clipped_left < SW) out.bend.top |= (unsigned int)(clipped_left + 1) << 20;
    out.line = line_of(clipped_left, clipped_right, clipped_dl, clipped_dr);
    return out;
}

// The same for a linedef's masked mid-texture, by four threads: its upper and lower edge, and the two ends of the sprite scale
// (engine.py:13480-13560).  `r` faces the camera with the side that carries the texture.
__device__ __forceinline__ void masked_lines(const DeviceMap &dm, const LaneCtx &c, const WallRec &r, int w, int k, MaskedGeo &out) {
    const gd_map_desc *m = &dm.d;
    const WallSide &ws = dm.wall_side[2 * w + ((r.flags & WF_FF) ? 0 : 1)];
    const float world_top = fminf(m->sector_heights[2 * m->wall_sectors[2 * w] + 1], m->sector_heights[2 * m->wall_sectors[2 * w + 1] + 1]);
    const HeightLine edge = height_line(c, r, (k & 1) ? world_top - (float)m->tex_h[ws.tex[0]] : world_top);
    i64 hoff, swall;
    texture_mapping(r, ws.repeat, (int)clampi((k & 1) ? r.sr - 1 : r.sl, 0, SW - 1), &hoff, &swall);
    i64 iscale = mul64(swall, FIXED_UNIT) >> 18;
    if (iscale >= 0 && iscale < 3) iscale = 3;
    else if (iscale > -3 && iscale < 0) iscale = -3;
    const i64 scale = tdiv(1LL << 32, iscale);
    const i64 other = (i64)(((u64)(unsigned)quad_move<0xB1>((int)(scale >> 32)) << 32) | (u64)(unsigned)quad_move<0xB1>((int)scale));
    if (k >= 2) return;
    out.line[k] = edge.line; out.bend[k] = edge.bend;
    if (bends(edge.bend)) out.outside[k] = edge.outside;
    if (k == 0) {
        out.scale.step = tdiv(other - scale, max64(r.sr - r.sl, 1));
        out.scale.base = (i64)((u64)scale - (u64)r.sl * (u64)out.scale.step);
    }
}

// A linedef's WallGeo by four threads of a quad: thread k takes height k.
__device__ __forceinline__ void wall_lines(const DeviceMap &dm, const LaneCtx &c, const WallRec &r, int w, int k, WallGeo &geo) {
    const gd_map_desc *m = &dm.d;
    const int sector = m->wall_sectors[2 * w + (k >> 1)];
    const float height = m->sector_heights[2 * (sector < 0 ? 0 : sector) + ((k == 0 || k == 3) ? 1 : 0)];
    const HeightLine line = height_line(c, r, height);
    geo.line[k] = line.line; geo.bend[k] = line.bend;
    if (bends(line.bend)) geo.outside[k] = line.outside;
    // the wallscan light (engine.py:11217-11291): thread k takes end k & 1 of side k >> 1
    const int side = k >> 1, end = k & 1;
    const i64 tx1 = side ? r.tx1 : r.tx0, tx2 = side ? r.tx0 : r.tx1, ty1 = side ? r.ty1 : r.ty0, ty2 = side ? r.ty0 : r.ty1;
    const i64 center = 160 * FIXED_UNIT;
    const i64 tx = end ? tx2 : tx1, ty = end ? ty2 : ty1;
    const bool inside = end ? tx2 <= ty2 : tx1 >= -ty1;
    const i64 projected = ((center + tdiv(tx * center, ty == 0 ? 1 : ty)) >> 16) + (tx >= 0);
    const i64 den = end ? ty2 - ty1 - tx2 + tx1 : tx1 - tx2 - ty2 + ty1;
    const i64 column = inside ? projected : (end ? SW : 0);
    const i64 depth = inside ? ty : ty1 + tdiv((ty2 - ty1) * (end ? tx1 - ty1 : tx1 + ty1), den == 0 ? 1 : den);
    const i64 light = tdiv(WALL_VISIBILITY_FIXED << 12, max64(depth, 1));
    auto other_end = [](i64 v) { return (i64)(((u64)(unsigned)quad_move<0xB1>((int)(v >> 32)) << 32) | (u64)(unsigned)quad_move<0xB1>((int)v)); };
    const i64 other_light = other_end(light), other_column = other_end(column);
    const i64 light_left = end ? other_light : light, light_right = end ? light : other_light;
    const i64 left = end ? other_column : column, right = end ? column : other_column;
    ColumnLine visibility;
    visibility.step = tdiv(light_right - light_left, max64(right - left, 1));
    visibility.base = (i64)((u64)light_left - (u64)left * (u64)visibility.step);
    if (end == 0) geo.visibility[side] = visibility;
    if (k == 0) {
        const bool spans = r.sr > r.sl;
        geo.tx0 = r.tx0; geo.tx1 = r.tx1; geo.ty0 = r.ty0; geo.ty1 = r.ty1;
        geo.span0 = (int)(spans ? clampi(r.sl, 0, SW) : 0); geo.span1 = (int)(spans ? clampi(r.sr, 0, SW) : 0);
        geo.past_left = r.sl > 0 ? 1 : 0;
    }
}

// The linedefs that the recorded passes of a lane draw, each worked out once (WallGeo) for all the columns and passes that draw it.
// The drawing half used to do this per column and pass: some 25 64-bit divisions, two thirds of its instructions, for what is
// the same in every column of a linedef.  `parts` (a power of two) work-groups of one wavefront a lane, none of which waits for another: each goes
// over the bits wall_select_kernel left, takes every parts-th group of sixteen of the linedefs they name, and gives four threads to a
// linedef (one a height; the wallscan light's four ends likewise).  Five more take a strip of columns each: masked mid-textures and the passes
// with rows of their own.  4096 lanes on the 4000-linedef map draw 1.3 million linedefs: 0.34 ms by one work-group a lane, whose 320 threads
// waited at barriers for the slowest, 0.29 by wavefronts that do strips after linedefs, 0.24 side by side in work-groups of four, 0.226 now;
// 512 lanes 0.084 -> 0.045, 16 lanes of the 320-linedef map 0.012 -> 0.008.  It waits for records and heights, then for its stores.
#define GEO_LIST 64                              // linedefs a wavefront lists at a time
template <bool SPLIT>
__global__ void __launch_bounds__(64) wall_geometry_kernel(DeviceMap dm, int lane_count, Scratch sc, int parts) {
    const gd_map_desc *m = &dm.d;
    __shared__ unsigned short list[GEO_LIST], masked_list[64];
    const int slot = threadIdx.x, k = slot & 3, quad = slot >> 2, shift = __ffs(parts) - 1;
    const int part = blockIdx.x, local = blockIdx.y;
    if (local >= lane_count) return;
    const LaneCtx &c = sc.ctx[local];
    const WallRec *recs = sc.rec + (size_t)local * m->wall_count;
    unsigned int *slots = sc.geo_slot + (size_t)local * m->wall_count;
    const unsigned int *named = sc.named + (size_t)local * named_words(m);
    const unsigned int first_slot = (unsigned)local * (unsigned)m->wall_count;   // the lane's run of geo
    const int words = named_words(m);
    if (part < parts) for (int pass = 0;; ++pass) {   // one, but for lanes that draw more than GEO_LIST * parts linedefs
        int total = 0;
        for (int word0 = 0; word0 < words; word0 += 64) {
            unsigned int bits = word0 + slot < words ? named[word0 + slot] : 0u;
            const int mine = __popc(bits);
            int upto = mine;
#pragma unroll
            for (int step = 1; step < 64; step <<= 1) { const int left = __shfl_up(upto, step); upto += slot >= step ? left : 0; }
            for (int rank = total + upto - mine; bits; bits &= bits - 1u, ++rank) {
                const int group = rank >> 4, at = (group >> shift) * 16 + (rank & 15) - pass * GEO_LIST;
                if ((group & (parts - 1)) == part && (unsigned)at < GEO_LIST) list[at] = (unsigned short)((word0 + slot) * 32 + __ffs((int)bits) - 1);
            }
            total += bcast(upto, 63);
        }
        wave_lds_fence();
        for (int j = 0; j < GEO_LIST / 16; ++j) {
            const int rank0 = ((pass * (GEO_LIST / 16) + j) * parts + part) * 16;
            if (rank0 >= total) break;            // the same in the whole wavefront
            if (rank0 + quad < total) {           // the four threads of a linedef are one DPP quad
                const int w = list[j * 16 + quad];
                const unsigned int at = first_slot + (unsigned)(rank0 + quad);
                wall_lines(dm, c, recs[w], w, k, sc.geo[at]);
                if (k == 0) slots[w] = at;
            }
        }
        if (((pass + 1) * (GEO_LIST / 16) * parts + part) * 16 >= total) return;
        wave_lds_fence();
    }
    {   // the other wavefronts: a strip of columns each
        const int strip = part - parts, x = strip * 64 + slot;
        if (dm.masked_count > 0) {
            // masked mid-textures: the linedef of every column's nearest one (its light and its texture mapping are WallGeo's)
            const u64 hit = sc.masked_hit[(size_t)local * SW + x];
            const int w = cand_key_wall(hit);
            // runs of columns share theirs: the first of a run (within its 16 columns) lists it
            const bool lists_it = hit != CAND_KEY_NONE && __builtin_amdgcn_update_dpp(-1, w, 0x111 /* row_shr:1 */, 0xF, 0xF, false) != w;
            const u64 listing = __ballot(lists_it);
            wave_lds_fence();
            if (lists_it) masked_list[__popcll(listing & ((1ULL << slot) - 1))] = (unsigned short)w;
            wave_lds_fence();
            MaskedGeo *masked = sc.masked_geo + (size_t)local * dm.masked_count;
            for (int entry = quad; entry < __popcll(listing); entry += 16) {
                const int mw = masked_list[entry];
                masked_lines(dm, c, recs[mw], mw, k, masked[dm.masked_slot[mw]]);
            }
        }
        // the few passes whose rows are their own, column by column
        if (!((sc.own_rows[local] >> strip) & 1u)) return;
        const WallRec *frags = sc.frag_rec + (size_t)local * m->split_count * m->fragment_slots;
        const int passes = sc.pass_count[(size_t)local * SW + x];
        PassRec next = {};
        if (passes > 0) next = sc.pass_rec[sc.pass_at(0, local, x)];
        for (int pass = 0; pass < passes; ++pass) {
            const size_t at = sc.pass_at(pass, local, x);
            const PassRec rec = next;
            if (pass + 1 < passes) next = sc.pass_rec[sc.pass_at(pass + 1, local, x)];
            if (!(rec.bits & (PB_RASTER | PB_PS_KEEPS)) || !(rec.marks & REC_OWN_ROWS)) continue;
            const int other = m->wall_sectors[2 * rec.wall + ((rec.marks & REC_SIDE1) ? 0 : 1)];
            unsigned int rows[2] = {0u, 0u};
#pragma unroll 1
            for (int h = 0; h < 8; ++h) {
                if (h < 4 ? (h >= 2 && (rec.bits & PB_ONE_SIDED)) : !(rec.bits & PB_PS_KEEPS)) continue;
                const int w = h < 4 ? rec.wall : rec.ps_path;
                const int behind = h < 4 ? other : (int)rec.ps_other;
                const int sector = (h & 2) ? (behind < 0 ? 0 : behind) : (int)rec.render_current;
                const float z = m->sector_heights[2 * sector + ((h & 3) == 0 || (h & 3) == 3 ? 1 : 0)];
                const FragmentChoice fragment = choose_fragment<SPLIT>(m, frags, recs[w], w, x);
                const unsigned int row = (unsigned int)project(c, recs[w], fragment, z, x);
                rows[h >> 2] |= row << (8 * (h & 3));
            }
            sc.pass_rows[at] = make_uint2(rows[0], rows[1]);
        }
    }
}

// How long a column's traversal runs is set by the portals it crosses: the two-sided linedefs its ray hits before the
// nearest blocking one.  Columns differ by a factor of ten, a wavefront runs as long as its longest column, and a launch
// ends with its longest wavefront.  So the screen is cut into segments of SEG_COLS columns, a wavefront takes
// 64 / SEG_COLS segments of about the same length (whatever lanes they belong to), and the longest go first.  The length
// is taken to be the longest candidate list of the segment, which wall_setup_kernel has counted anyway: walking the lists
// to count the portals proper orders the segments a little better (the traversal gains 0.04 ms on the 4000-linedef map)
// but the walk costs 0.11 ms.  wall_setup_kernel or strip_key_kernel takes the maxima, strip_order_kernel sorts them (one block, counting sort).
// Narrow segments waste fewer column passes (on the 4000-linedef map 69 % of the passes a wavefront runs are useful with
// whole 64-column strips, 80 % with two sorted 32-column segments, 89 % with four of 16), but unrelated segments share no
// linedefs, branches or row ranges, and a pass costs what the union of its columns' paths costs: measured, the traversal
// takes 3.86 ms with 64 or 32 columns a segment, 4.06 ms with 16 and 4.23 ms with 8.  Hence whole strips.
__global__ void __launch_bounds__(256) strip_key_kernel(int lane_count, Scratch sc) {   // of lanes whose linedefs were dealt out (wall_setup_kernel)
    const int strip = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int local = strip / (SW / 64);
    if (local >= lane_count) return;
    const int x = (strip - local * (SW / 64)) * 64 + (threadIdx.x & 63);
    note_length(sc, local, x, sc.cand_count[(size_t)local * SW + x]);
}

#define SPILL_BLOCKS 64
__global__ void __launch_bounds__(1024) strip_order_kernel(DeviceMap dm, int strips, Scratch sc) {
    if (blockIdx.x > 0) {        // the others list the spilled columns afresh
        list_spilled_columns(dm, sc, (blockIdx.x - 1) * 16 + (threadIdx.x >> 6), (gridDim.x - 1) * 16);
        return;
    }
    __shared__ int histogram[CAND_MAX + 1], position[CAND_MAX + 1];
    for (int k = threadIdx.x; k <= CAND_MAX; k += blockDim.x) histogram[k] = 0;
    __syncthreads();
    for (int s = threadIdx.x; s < strips; s += blockDim.x) atomicAdd(&histogram[sc.strip_key[s]], 1);
    __syncthreads();
    if (threadIdx.x == 0) {
        int running = 0;
        for (int k = CAND_MAX; k >= 0; --k) { position[k] = running; running += histogram[k]; }
    }
    __syncthreads();
    for (int s = threadIdx.x; s < strips; s += blockDim.x) sc.strip_order[atomicAdd(&position[sc.strip_key[s]], 1)] = s;
}

// The traversal in two kernels.  Which drawseg a column pass selects, and where the column goes next, depends on the map,
// the camera and the column's ray alone, never on projected rows or clips: wall_select_kernel runs that half
// (pass_select without the projection, pass_advance) and records one PassRec per pass; wall_raster_kernel
// runs the other half over the records (pass_draw, clip_pass, pass_paint, advance_clips, the masked mid-texture).
// Each half is lighter in registers and in code than the two together, so more of its wavefronts share a SIMD and
// its pass loop fits the instruction cache.  Same segment order and one wavefront per segment in both.
// The kernel lasts as long as its longest strips.  Such a strip's wavefront is held up by its candidate scans (the longest lists) and by running,
// pass after pass, every rule that any of its 64 columns takes.  So in the longest strips (they lead the order; select_strips) a column has LANES
// lanes: a strip is LANES wavefronts, the lanes of a
// column hold its list between them in registers, each scans its own entries, and what a scan is after is the smallest of the lanes' keys, three to
// five lane moves away.  All else they do alike, and the first of them writes the records.  The stage with a lane a column in all strips, and with these shared out:
// 64 lanes on the 2000-linedef map 216, 66 us, 512 lanes of it 256, 125; on the 4000-linedef map 64 lanes 372, 89, 512 lanes 470, 173, 4096 lanes 782, 564.  What the
// rules ask beyond the list (a sector bridge) they ask behind the scan, once for each entry concerned: a copy of that code for every entry made the
// kernels larger than the instruction cache.
static_assert(SEG_COLS == 64, "wall_select_kernel: a work-group is one wavefront, with columns of one strip");
// The columns of one wavefront: 64 / LANES of a strip's, from the `part`-th such share on.
template <bool SPLIT, int LANES>
__device__ __forceinline__ void select_columns(const DeviceMap &dm, const Scratch &sc, const LaneCtx &lane_ctx, unsigned *window_lds, int local, int strip_x, int part) {
    const gd_map_desc *m = &dm.d;
    constexpr bool SHARED = LANES > 1;
    constexpr int part_cols = 64 / LANES;
    const int lane_id = threadIdx.x & 63, lane_of_column = lane_id & (LANES - 1);
    const int x = strip_x + part * part_cols + lane_id / LANES;
    ColumnCtx cc;
    cc.tb = nullptr; cc.m = m; cc.mv.m = m; cc.mv.walls = dm.wall_links; cc.mv.vertex_links = dm.vertex_links; cc.c = &lane_ctx;
    cc.recs = sc.rec; cc.spans = sc.span;
    cc.rec_base = (unsigned)local * (unsigned)m->wall_count;
    cc.frags = sc.frag_rec + (size_t)local * m->split_count * m->fragment_slots;
    cc.set_list(sc, local, x);
    cc.x = x;
    ray_direction(lane_ctx, x, &cc.rx, &cc.ry);
    cc.first = cc.eval(0);
    bool boundary_has_po = false;   // does some entry's span begin at this column
    bool stand_in = false;          // does some entry show all of STANDS_IN
    ListShare<LANES> list;
    if constexpr (SHARED) {
        list.load(cc, lane_of_column);
        unsigned first = 3u;
        list.each(cc, [&](const ListEntry &q) { first &= ~(((q.flags & CF_LEDGE) ? 1u : 0u) | ((q.flags & STANDS_IN) == STANDS_IN ? 2u : 0u)); });
        boundary_has_po = list.smallest(first & 1u) == 0u; stand_in = list.smallest(first & 2u) == 0u;
    }
    ColumnState st;
    st.current_sector = lane_ctx.sector;
    st.ceiling_clip = 0.0f; st.floor_clip = (float)VH;
    st.masked_ceiling_clip = 0.0f; st.masked_floor_clip = (float)VH; st.masked_distance = GD_INF; st.masked_wall = -1;
    st.previous_distance = 0.0f;
    st.pend_po_vertex = -1; st.pend_ep_vertex = -1; st.pend_ep_wall = 0; st.pend_ep_sectors = 0; st.pend_ep_vertices = 0; st.pend_eb_index = 0;
    st.pend_pb_index = 0; st.pend_pb_sector = -1; st.pend_pb_exit = 0.0f; st.flags = 0;
    if constexpr (!SHARED) list.start(cc, window_lds, lane_id, boundary_has_po, stand_in);
    // A column that has come to the end of its way has no sector.  The passes that follow look at linedef 0 in place of a linedef and at sector 0 in place of
    // a sector.  They find nothing, draw nothing and change nothing but flags that only matter where something is found, unless a solid linedef of sector 0 begins at
    // the column, linedef 0's span ends at it, a neighbour of linedef 0 owns it, or an endpoint's boundary is still pending: but for these the column is done.
    bool ends_quietly = !stand_in && !(cc.first.flags & CF_ENDS_HERE);
    {
        int owner; Eval of_owner;
        endpoint_owner(cc, 0, cc.first, cc.mv.walls[0], &owner, &of_owner);
        ends_quietly = ends_quietly && owner == 0;
    }
    PassRec *records = sc.pass_rec + sc.pass_at(0, local, x);
    float *path_distances = sc.pass_path_distance + sc.pass_at(0, local, x);
    const size_t pass_stride = (size_t)sc.lane_stride * SW;
    // the linedefs the recorded passes draw get a bit each; columns that draw what the column before them draws leave it to that one
    unsigned int *named = sc.named + (size_t)local * named_words(m);
    int last_named = -1;
    auto neighbour = [](int v) { return LANES < 16 ? __builtin_amdgcn_update_dpp(-1, v, 0x110 + (LANES & 15) /* row_shr */, 0xF, 0xF, false) : -1; };
    if (dm.masked_count > 0) {   // so do those whose masked mid-texture is a column's nearest
        const u64 hit = sc.masked_hit[(size_t)local * SW + x];
        const int w = cand_key_wall(hit);
        const int left = neighbour(w);
        if (lane_of_column == 0 && hit != CAND_KEY_NONE && left != w) atomicOr(&named[w >> 5], 1u << (w & 31));
    }
    PassColumn pc;
    bool done = false;
    int recorded = 0;
    const int sectors = m->sector_count;
    for (int pass = 0; pass < sectors; ++pass) {
        if (!done) {
            pass_select<SPLIT>(cc, list, st, boundary_has_po, pc);
            if (pc.bits & (PB_RASTER | PB_PS_KEEPS)) {
                const bool repeats = last_named == pc.wall;
                last_named = pc.wall;
                // a neighbour that does not take part in this pass shows the linedef it named last
                const bool names = !repeats && neighbour(last_named) != last_named;
                if (lane_of_column != 0) {
                    recorded = pass + 1;
                } else if (pass < sc.pass_slots) {
                    PassRec rec;
                    rec.wall = (unsigned short)pc.wall; rec.render_current = (unsigned short)pc.render_current;
                    rec.bits = (unsigned short)pc.bits; rec.ps_path = (unsigned short)pc.ps_path_index;
                    rec.ps_other = (short)pc.ps_other; rec.marks = (unsigned short)pc.marks; rec.distance = pc.distance;
                    // passes between two recorded ones keep whatever the slot held: the drawing half skips them by their bits
                    for (int skipped = recorded; skipped < pass; ++skipped) records[(size_t)skipped * pass_stride].bits = 0;
                    records[(size_t)pass * pass_stride] = rec;
                    if (names) atomicOr(&named[pc.wall >> 5], 1u << (pc.wall & 31));
                    if (pc.bits & PB_PS_KEEPS) {
                        path_distances[(size_t)pass * pass_stride] = pc.ps_path_distance;
                        atomicOr(&named[pc.ps_path_index >> 5], 1u << (pc.ps_path_index & 31));
                    }
                    if (pc.marks & REC_OWN_ROWS) atomicOr(&sc.own_rows[local], 1u << (x >> 6));
                    recorded = pass + 1;
                } else {
                    sc.status[STATUS_PASS_OVERFLOW] = 1;
                }
            }
            const bool changed = pass_advance<SPLIT>(cc, list, st, pc);
            // A pass that found nothing and changed nothing repeats identically for ever.
            if (!(pc.bits & PB_VALID) && !changed) done = true;
            if (ends_quietly && st.current_sector < 0 && !(st.flags & ST_EP)) done = true;
        }
        if (__ballot(!done) == 0) break;
    }
    if (lane_of_column == 0) sc.pass_count[(size_t)local * SW + x] = (unsigned char)recorded;
}

// The strips from `first` on in the order: `longest` of them with LANES wavefronts each, and as many more of one wavefront, a lane a column, as the
// grid has wavefronts for.  The two kinds start by turns, eight wavefronts of each, so that both are dealt out over all eight dies and neither waits for
// the other's to end.  A strip of the longest that its lanes cannot hold is drawn here too, not in a launch behind this one, which small batches
// paid 7 us for.  (16 lanes: 130 registers left to itself, 128 as told.)
template <bool SPLIT, int LANES>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(LANES == 8 ? 3 : 4))) wall_select_kernel(DeviceMap dm, Scratch sc, int first, int longest) {
    __shared__ LaneCtx lane_ctx;
    __shared__ __align__(8) unsigned window_lds[ListShare<1>::WORDS];
    const int shares = longest * LANES, others = (int)gridDim.x - shares, mixed = min(shares, others) & ~7, b = (int)blockIdx.x;
    const bool beyond = b < 2 * mixed ? (b & 8) != 0 : shares - mixed <= b - 2 * mixed;
    const int at = b < 2 * mixed ? ((b >> 4) << 3) | (b & 7) : (beyond ? b - shares : b - mixed);
    const int segment = sc.strip_order[first + (beyond ? longest + at : at / LANES)], part = beyond ? 0 : at % LANES;
    const int local = segment / SEGS_PER_LANE, strip_x = (segment - local * SEGS_PER_LANE) * SEG_COLS;
    if (threadIdx.x == 0) lane_ctx = sc.ctx[local];
    __syncthreads();
    if constexpr (LANES > 1) {
        // A strip with a column in the spill pool (more entries than its lanes hold) is the first of its wavefronts', a lane a column.
        if (beyond || __ballot(((unsigned)sc.cand_count[(size_t)local * SW + strip_x + threadIdx.x] >> SPILL_SHIFT) != 0) != 0) {
            if (beyond || part == 0) select_columns<SPLIT, 1>(dm, sc, lane_ctx, window_lds, local, strip_x, 0);
            return;
        }
    }
    select_columns<SPLIT, LANES>(dm, sc, lane_ctx, window_lds, local, strip_x, part);
}

// One wavefront per 64 / SEG_COLS segments.  Segments share nothing but read-only tables; a work-group of the drawing
// half is WALL_STRIPS_PER_GROUP wavefronts (neighbours in the longest-first order) only so that the LDS copies of
// those tables, 16.7 KB, are held once per group rather than once per wavefront (a CU has 160 KB of LDS and room for
// sixteen of these wavefronts at 128 registers).  After the staging barrier the wavefronts never meet again.
#define WALL_STRIPS_PER_GROUP 2
static_assert(32 * 256 / 16 % (64 * WALL_STRIPS_PER_GROUP) == 0, "wall_raster_kernel: the colormap's rows in whole turns");
#define RASTER_WAVES 4
// The pass that the lane `k` of each column's PARTS lanes prepared, for all of them.
template <int PARTS>
__device__ __forceinline__ PassDraw hand_round(const PassDraw &prepared, int k, int lane_id) {
    if (PARTS == 1) return prepared;
    constexpr int COLUMNS = SEG_COLS / PARTS;
    const int from = (k * COLUMNS + (lane_id & (COLUMNS - 1))) * 4;
    auto take = [&](unsigned int v) { return (unsigned int)__builtin_amdgcn_ds_bpermute(from, (int)v); };
    PassDraw d;
    d.flags = take(prepared.flags); d.wall_sector = take(prepared.wall_sector); d.rows = take(prepared.rows);
    d.column_a = take(prepared.column_a); d.frac_a = take(prepared.frac_a); d.step_a = take(prepared.step_a);
    d.column_b = take(prepared.column_b); d.frac_b = take(prepared.frac_b); d.step_b = take(prepared.step_b);
    d.distance = __uint_as_float(take(__float_as_uint(prepared.distance)));
    return d;
}
// DEPTH: also keep the depth of every wall pixel (frames that draw decals).  GENERAL: the map has linedefs with
// BSP projection fragments, or more sectors or textures than the LDS tables hold (a table that may be in either place is read
// behind a branch, and behind a branch with a load in it a wavefront waits for every store it has under way).
// 4096 lanes on the 4000-linedef map: 1.78 -> 1.00 ms: the linedefs' lines 1.53, no sprite clip plane
// and the rows walked together 1.33, no branch around a load or a store 1.03.  It is left at four wavefronts a SIMD (128 registers;
// at 96 the spills in the row loops make it 1.6 ms), 60 % of their cycles waiting.  By itself, with a column's lanes sharing its passes and
// rows: 16 lanes on the 2000-linedef map 97 -> 53 us, 512 on the 4000-linedef map 443 -> 350, 1024 on the 320-linedef map 286 -> 226 (rows alone
// 71, 426, 252).  The passes are handed round from register to register: through LDS there are no spills, but the 1024 lanes take 268.  Working
// out the textures of visible tiers only makes the 1024 lanes 241, and 4096 1.11 ms.
template <bool DEPTH, bool GENERAL, int PARTS>
__global__ void __launch_bounds__(64 * WALL_STRIPS_PER_GROUP) __attribute__((amdgpu_waves_per_eu(RASTER_WAVES, RASTER_WAVES))) wall_raster_kernel(DeviceMap dm, int lane_count, Scratch sc, unsigned char *frame_base, size_t frame_stride) {
    const gd_map_desc *m = &dm.d;
    __shared__ LaneCtx lane_ctxs[WALL_STRIPS_PER_GROUP][64 / SEG_COLS];
    __shared__ __align__(16) unsigned char colormap_lds[32 * 256];   // shade rows 0..31 are the only ones indexed
    __shared__ float4 sector_lds[LDS_SECTORS];
    __shared__ TexLds tex_lds;
    const int wave_in_group = threadIdx.x >> 6;
    const int lane_id = threadIdx.x & 63;
    const int segment_in_wave = lane_id / SEG_COLS;
    const int wavefront = blockIdx.x * WALL_STRIPS_PER_GROUP + wave_in_group;
    constexpr int part_cols = SEG_COLS / PARTS;
    const int segment_slot = wavefront / PARTS, part = wavefront % PARTS;
    const bool live = segment_slot < lane_count * SEGS_PER_LANE;
    const int segment = live ? sc.strip_order[segment_slot] : 0;
    const int local = segment / SEGS_PER_LANE;
    Tables tb;
    stage_tables(m, sector_lds, &tex_lds, tb);
    tb.all_cached = !GENERAL;
    if ((lane_id & (SEG_COLS - 1)) == 0 && live) lane_ctxs[wave_in_group][segment_in_wave] = sc.ctx[local];
#pragma unroll
    for (int k = 0; k < 32 * 256 / 16; k += 64 * WALL_STRIPS_PER_GROUP) reinterpret_cast<uint4 *>(colormap_lds)[k + threadIdx.x] = reinterpret_cast<const uint4 *>(m->colormap)[k + threadIdx.x];
    __syncthreads();
    if (!live) return;   // whole segments: the groups of four columns that exchange values below live or leave together
    const LaneCtx &lane_ctx = lane_ctxs[wave_in_group][segment_in_wave];
    // a wavefront's part_cols columns have `parts` lanes each, which do everything alike and share the rows out
    const bool own_column = lane_id < part_cols;
    const int x = (segment - local * SEGS_PER_LANE) * SEG_COLS + part * part_cols + (lane_id & (part_cols - 1));
    bool window_dirty = false;
    GapRange gaps; gaps.reset();
    ColumnCtx cc;
    cc.tb = &tb; cc.m = m; cc.c = &lane_ctx;
    cc.recs = sc.rec; cc.spans = sc.span;
    cc.rec_base = (unsigned)local * (unsigned)m->wall_count;
    cc.frags = sc.frag_rec + (size_t)local * m->split_count * m->fragment_slots;
    cc.x = x;
    ray_direction(lane_ctx, x, &cc.rx, &cc.ry);
    PixelBuffers<PARTS> pb;
    pb.meta = sc.meta;
    pb.scene_depth = DEPTH ? sc.scene_depth : nullptr;
    pb.word_column = ((unsigned)local * (VH * SW) + (unsigned)x) * 4u;
    pb.words = __builtin_amdgcn_make_buffer_rsrc(sc.meta, 0, lane_count * (VH * SW * 4), BUFFER_WORDS);
    pb.depths = __builtin_amdgcn_make_buffer_rsrc(pb.scene_depth, 0, DEPTH ? lane_count * (VH * SW * 4) : 0, BUFFER_WORDS);
    pb.row_lane = PARTS == 1 ? 0 : lane_id / part_cols;
    const unsigned byte_stride = frame_base ? (unsigned)frame_stride : VH * SW;
    pb.bytes = __builtin_amdgcn_make_buffer_rsrc(frame_base ? frame_base : sc.masked_texel, 0, (frame_base || sc.masked_texel) ? lane_count * (int)byte_stride : 0, BUFFER_WORDS);
    pb.put_byte_column = (unsigned)local * byte_stride + (unsigned)pb.row_lane * SW + (unsigned)x;
    pb.put_column = pb.word_column + (unsigned)pb.row_lane * (SW * 4u);
    // the meta plane arrives with whatever the last frame left: see GapRange for how every row gets written
    ColumnState st;   // only the clips and the masked-drawseg snapshot live here; the traversal state stayed in wall_select_kernel
    st.current_sector = -1;
    st.ceiling_clip = 0.0f; st.floor_clip = (float)VH;
    st.masked_ceiling_clip = 0.0f; st.masked_floor_clip = (float)VH; st.masked_distance = GD_INF; st.masked_wall = -1;
    st.previous_distance = 0.0f;
    st.pend_po_vertex = -1; st.pend_ep_vertex = -1; st.pend_ep_wall = 0; st.pend_ep_sectors = 0; st.pend_ep_vertices = 0; st.pend_eb_index = 0;
    st.pend_pb_index = 0; st.pend_pb_sector = -1; st.pend_pb_exit = 0.0f; st.flags = 0;
    SilhouetteBounds sb; sb.bot_row = VH; sb.top_row = 0; sb.bot_depth = -GD_INF; sb.top_depth = -GD_INF; sb.deepest = -GD_INF;
    const int passes = sc.pass_count[(size_t)local * SW + x];
    const size_t first_record = sc.pass_at(0, local, x), pass_stride = (size_t)sc.lane_stride * SW;
    const unsigned int *geo_slots = sc.geo_slot + cc.rec_base;
    // Each of a column's lanes prepares every PARTS-th pass, so that what a pass has to ask memory for is on its way for PARTS of them
    // at once; then the passes are drawn one after the other, each handed round from the lane that prepared it.
    // A pass's record names its linedef, the linedef's slot where it lies in geo: the next pass's slot and the record after it
    // are asked for a pass ahead.  (Columns past their last pass keep asking for their first one.)
    PassRec record = {}, next_record = {};
    unsigned int slot = 0u, slot_wall = 0u;      // a pass that draws nothing names no linedef: the slot of the last one asked for will do
    const size_t group_stride = PARTS * pass_stride;
    size_t prepared_at = first_record + (size_t)pb.row_lane * pass_stride;
    if (passes > 0) {
        record = sc.pass_rec[pb.row_lane < passes ? prepared_at : first_record]; next_record = sc.pass_rec[pb.row_lane + PARTS < passes ? prepared_at + group_stride : first_record];
        slot_wall = record.bits ? record.wall : 0u;
        slot = geo_slots[slot_wall];
    }
    for (int group = 0; __ballot(group < passes) != 0; group += PARTS) {
        const int pass = group + pb.row_lane;
        const PassRec rec = record;
        unsigned int geo_at = slot;
        if (group < passes) {
            if constexpr (PARTS == 1) {
                record = next_record;
                slot_wall = record.bits ? record.wall : slot_wall;
                slot = geo_slots[slot_wall];
                next_record = sc.pass_rec[pass + 2 * PARTS < passes ? prepared_at + 2 * group_stride : first_record];
            } else {
                geo_at = geo_slots[rec.bits ? rec.wall : 0];
                record = sc.pass_rec[pass + PARTS < passes ? prepared_at + group_stride : first_record];
            }
        }
        const PassDraw prepared = pass_draw<GENERAL>(dm, cc, sc, pass < passes && (rec.bits & (PB_RASTER | PB_PS_KEEPS)) != 0, rec, geo_at, prepared_at);
        prepared_at += group_stride;
#pragma unroll 1
        for (int k = 0; k < PARTS; ++k) {
            if (PARTS > 1 && __ballot(group + k < passes) == 0) break;
            const PassDraw d = hand_round<PARTS>(prepared, k, lane_id);
            const PassRows rows = clip_pass(d, st.ceiling_clip, st.floor_clip);
            // The aligned group of four columns agrees on which tiers all four draw and on the rows all four share: minima, maxima and
            // conjunctions over the quad take two steps each.  Every lane of the wavefront is active here.
            const bool raster = d.flags & DRAW_RASTER, one_sided = d.flags & DRAW_ONE_SIDED, texture_a = d.flags & DRAW_TEXTURE_A;
            const bool tier0 = raster && one_sided && texture_a && rows.top < rows.bottom;
            const bool tier1 = raster && (d.flags & DRAW_LOWER) && texture_a && rows.lower_top < rows.bottom;
            const bool tier2 = raster && (d.flags & DRAW_UPPER) && (d.flags & DRAW_TEXTURE_B) && rows.top < rows.upper_bottom;
            const int agreed = quad_and((tier0 ? 1 : 0) | (tier1 ? 2 : 0) | (tier2 ? 4 : 0));
            const bool same_group = d.flags & DRAW_GROUP;
            const float shared_top = quad_max(rows.top), shared_lower_top = quad_max(rows.lower_top);
            const float shared_bottom = quad_min(rows.bottom), shared_upper_bottom = quad_min(rows.upper_bottom);
            const float common_bottom[3] = {shared_bottom, shared_bottom, shared_upper_bottom};
            bool group_valid[3];
            group_valid[0] = same_group && (agreed & 1) && (shared_top < shared_bottom);
            group_valid[1] = same_group && (agreed & 2) && (shared_lower_top < shared_bottom);
            group_valid[2] = same_group && (agreed & 4) && (shared_top < shared_upper_bottom);
            pass_paint<DEPTH>(cc, st, d, rows, pb, group_valid, common_bottom, colormap_lds, window_dirty, gaps);
            advance_clips(cc, st, d, rows, pb, sb, !window_dirty, gaps, sc, first_record + (size_t)(group + k) * pass_stride);
        }
    }
    // what is left of a window no one-sided drawseg closed shows the flat pass's picture
    if (!window_dirty) zero_rows(pb, gaps, x, st.ceiling_clip <= 0.0f ? 0 : (int)st.ceiling_clip, st.floor_clip >= (float)VH ? VH : (int)st.floor_clip);
    if (dm.masked_count > 0) masked_midtexture<DEPTH, GENERAL>(dm, cc, sc, local, st, pb, colormap_lds);
    // The columns with view pixels that no wall tier, plane or masked texture covers join the flat pass's work list, those of a
    // wavefront in one piece (flat_gap_kernel selects the pixels, flat_shade_kernel paints them).
    bool holds_gap = false;
    wave_fence();
    for (int y = gaps.lo() + pb.row_lane, gap_end = gaps.hi(); y < gap_end && !holds_gap; y += PARTS) holds_gap = gap_pixel(pb.m(y));
    u64 holders = __ballot(holds_gap);
    if (holders == 0) return;
    for (int other = 32; other >= part_cols; other >>= 1) holders |= holders >> other;   // a column's lanes
    holders &= ~0ULL >> (64 - part_cols);
    holds_gap = own_column && (holders >> lane_id & 1);
    int list_base = 0;
    if (lane_id == 0) list_base = atomicAdd(sc.gap_column_count, __popcll(holders));
    list_base = __builtin_amdgcn_readfirstlane(list_base);
    if (holds_gap) sc.gap_columns[list_base + __popcll(holders & ((1ULL << lane_id) - 1))] = make_int2((local << 9) | x, gaps.lo() | (gaps.hi() << 8));
}

// ---------------------------------------------------------------------------------------------
// plane shading.  A pixel no wall tier owns shows a flat: the visplane the wall traversal marked for it (engine.py:13372-13405)
// or, where no drawseg marked one, the sector the per-pixel plane rays selected (engine.py:11145-11163).  Doing the first for every
// pixel here and the second in flat_shade_kernel shades every pixel once.
// ---------------------------------------------------------------------------------------------
// A wavefront takes a tile of 64 columns and SHADE_ROWS rows, a column a lane.  Everything but the texel is the same along a run of
// pixels of a row that show one plane: each run's leftmost pixel is listed, a lane works out each listed run (PlaneSpan, one pass for
// up to 64 of them: a tile has some forty), and its pixels read it back from LDS.  Bound by the per-pixel words in and the pixels out (1.4 GB at 4096
// lanes, 4.1 of the 5.2 TB/s of a copy), then by its vector instructions; a work-group is four tiles (all of a lane's by two work-groups: 0.41 ms,
// five tiles 0.44, stores of four columns' words 0.54).  4096 lanes on the 4000-linedef map: 0.69 ms with a run of four pixels a thread (each plane
// of the four worked out again), 0.374 at 717 vector instructions a tile, 0.342 now at 533 (the compiler's 32-bit multiplications as 24-bit ones,
// no branch a pixel, a run's number that needs no range test); 16 lanes 0.043, 0.010, 0.009.
#define SHADE_ROWS 16
#define SHADE_BATCH 4        // rows whose texels are asked for together
#define RUN_NONE 0x7FFu      // the number of a pixel's run, or that it has none (a tile has at most 1024)
#define RUN_ROUND 0x7C0u     // the first run of the round that works it out
#define SHADE_THREADS 256
#define SHADE_TILES ((SW / 64) * (VH / SHADE_ROWS))      // a lane's; a wavefront takes one
static_assert(SW % 64 == 0 && VH % SHADE_ROWS == 0 && SHADE_ROWS <= 16, "plane_shade_kernel: whole tiles, of at most 1024 runs");
static_assert((GD_SCREEN_HEIGHT - VH) * SW / 4 <= SHADE_TILES * 64, "plane_shade_kernel: a tile clears a word of the status bar a lane");
__global__ void __launch_bounds__(SHADE_THREADS) __attribute__((amdgpu_waves_per_eu(8, 8))) plane_shade_kernel(DeviceMap dm, int lane_count, Scratch sc, unsigned char *frame_base, size_t frame_stride) {
    const gd_map_desc *m = &dm.d;
    constexpr int WAVES = SHADE_THREADS / 64;
    __shared__ __align__(16) unsigned char colormap_lds[32 * 256];
    struct Runs { uint4 start[64], step[64]; unsigned int texture[64]; };      // a listed run in `texture`, until its lane puts the run's texture there
    __shared__ Runs runs_lds[WAVES];
    const int local = blockIdx.y;
    if (local >= lane_count) return;     // uniform over the block
    const LaneCtx &c = sc.ctx[local];
    const int lane_id = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Runs &runs = runs_lds[wave];
    unsigned char *frame = frame_base + (size_t)local * frame_stride;
    // the lane's words and view pixels as buffers: a pixel that is not this kernel's is stored beyond the end, which the hardware drops
    // (with a branch around every store the rows' addresses and masks alone would fill the registers)
    const __amdgpu_buffer_rsrc_t words = __builtin_amdgcn_make_buffer_rsrc(sc.meta + (size_t)local * VH * SW, 0, VH * SW * 4, BUFFER_WORDS);
    const __amdgpu_buffer_rsrc_t pixels = __builtin_amdgcn_make_buffer_rsrc(frame, 0, VH * SW, BUFFER_WORDS);
    const unsigned atlas_width = (unsigned)m->tex_max_w;
    // what names a pixel's plane in its word: the sector and which of its two planes
    const unsigned int PLANE_KEY = (META_SECTOR_MASK << META_SECTOR_SHIFT) | META_FLOOR;
    const int tile = blockIdx.x * WAVES + wave, x_first = tile % (SW / 64) * 64, y_first = tile / (SW / 64) * SHADE_ROWS;
    const unsigned at = (unsigned)(y_first * SW + x_first + lane_id);
    auto put = [&](bool own, int r, unsigned colour) { __builtin_amdgcn_raw_buffer_store_b8((unsigned char)colour, pixels, own ? at : BUFFER_NOWHERE, r * SW, 0); };
    unsigned int meta[SHADE_ROWS];
#pragma unroll
    for (int r = 0; r < SHADE_ROWS; ++r) meta[r] = __builtin_amdgcn_raw_buffer_load_b32(words, at * 4u, r * (SW * 4), 0);
    for (int k = threadIdx.x; k < 32 * 256 / 16; k += SHADE_THREADS) reinterpret_cast<uint4 *>(colormap_lds)[k] = reinterpret_cast<const uint4 *>(m->colormap)[k];
    __syncthreads();
    if (tile < (GD_SCREEN_HEIGHT - VH) * SW / 4 / 64) {   // the empty status bar, rows 208..239
        unsigned char *bar = frame + (size_t)VH * SW + (size_t)(tile * 64 + lane_id) * 4;
        if ((reinterpret_cast<size_t>(frame) & 3) == 0) *reinterpret_cast<unsigned int *>(bar) = 0u;
        else for (int k = 0; k < 4; ++k) bar[k] = 0;
    }
    if (tile >= SHADE_TILES) return;     // the last work-group's spare wavefronts; their words lay beyond the buffer
    // Each pixel's word becomes: what names its plane and the number of its run; or a tier's colour and RUN_NONE.
    int total = 0;
#pragma unroll
    for (int r = 0; r < SHADE_ROWS; ++r) {
        // no run where no plane shows (a wall tier, a masked texture, or neither tier nor plane: the flat pass's picture, which
        // flat_shade_kernel paints once that pass has run)
        const unsigned int word = (meta[r] & META_MASKED) ? 0u : meta[r] & (META_FILLED | PLANE_KEY);
        const unsigned int key = (unsigned)max((int)word, 0);      // a tier's word is negative, that of neither tier nor plane is zero
        const unsigned int left = (unsigned)__builtin_amdgcn_update_dpp(0, (int)key, 0x138 /* wave_shr:1 */, 0xF, 0xF, true);
        const bool plane = key != 0u;
        const u64 begins = __builtin_amdgcn_ballot_w64(plane) & __builtin_amdgcn_ballot_w64(key != left), before = begins >> 1;
        const int run = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(before >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)before, 0u)) + (total + (int)(begins & 1) - 1);
        meta[r] = word | (plane ? (unsigned)run : RUN_NONE);
        if (__builtin_amdgcn_inverse_ballot_w64(begins) && run < 64) runs.texture[run] = key | (unsigned)r;
        total += __popcll(begins);
    }
    for (unsigned first = 0;;) {     // one round, but for the most varied tiles
        wave_lds_fence();
        {
            PlaneSpan span = {};                 // lanes without a run leave one whose texel is the atlas's first: pixels without one ask for it
            if (first + lane_id < (unsigned)total) {
                const unsigned int listed = runs.texture[lane_id];
                span = plane_span(dm, sc, c, local, (int)((listed >> META_SECTOR_SHIFT) & META_SECTOR_MASK) - 1, (listed & META_FLOOR) != 0, x_first, y_first + (int)(listed & 0xFFFFu));
            }
            runs.start[lane_id] = span.start; runs.step[lane_id] = span.step; runs.texture[lane_id] = span.texture;
        }
        wave_lds_fence();
#pragma unroll
        for (int r0 = 0; r0 < SHADE_ROWS; r0 += SHADE_BATCH) {
            bool here[SHADE_BATCH], any = false;     // is the pixel's run one of this round's
#pragma unroll
            for (int j = 0; j < SHADE_BATCH; ++j) { here[j] = (meta[r0 + j] & RUN_ROUND) == first; any |= here[j]; }
            if (__any(any)) {
                unsigned shade_at[SHADE_BATCH]; unsigned char texel[SHADE_BATCH];
#pragma unroll
                for (int j = 0; j < SHADE_BATCH; ++j) {
                    const unsigned run = meta[r0 + j] & 63u;
                    PlaneSpan span;
                    span.start = runs.start[run]; span.step = runs.step[run]; span.texture = runs.texture[run];
                    texel[j] = m->tex_atlas[span.texel((unsigned)lane_id, atlas_width)];
                    shade_at[j] = span.colormap_row() * 256;
                }
                __builtin_amdgcn_sched_barrier(0);   // all of the batch's texels are asked for before the first is looked at
#pragma unroll
                for (int j = 0; j < SHADE_BATCH; ++j) {
                    unsigned colour = colormap_lds[shade_at[j] + texel[j]];
                    asm volatile("" : "+v"(colour));   // looked up for all pixels: a branch around it costs more
                    const bool tier = (int)meta[r0 + j] < 0;
                    put(here[j] || (tier && first == 0), r0 + j, tier ? meta[r0 + j] >> META_SECTOR_SHIFT : colour);
                }
            } else if (first == 0) {
#pragma unroll
                for (int j = 0; j < SHADE_BATCH; ++j) put((int)meta[r0 + j] < 0, r0 + j, meta[r0 + j] >> META_SECTOR_SHIFT);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        first += 64;
        if (first >= (unsigned)total) break;
        wave_lds_fence();
#pragma unroll
        for (int r = 0; r < SHADE_ROWS; ++r) {
            asm volatile("" : "+v"(meta[r]));      // worked on afresh in every round: kept over the rounds, its derivatives would fill the registers
            const unsigned int left = (unsigned)__builtin_amdgcn_update_dpp((int)RUN_NONE, (int)meta[r], 0x138 /* wave_shr:1 */, 0xF, 0xF, false);
            const unsigned run = (meta[r] & RUN_NONE) - first;
            if (((left ^ meta[r]) & RUN_NONE) && run < 64u) runs.texture[run] = (meta[r] & PLANE_KEY) | (unsigned)r;
        }
    }
}

// The listed gap pixels, painted with the flat the flat pass settled on (engine.py:11145-11163).
__device__ void flat_shade_pixel(const DeviceMap &dm, const Scratch &sc, const LaneCtx &c, int local, int pixel, unsigned char *frame) {
    const gd_map_desc *m = &dm.d;
    Tables tb; tb.m = m; tb.sector = nullptr; tb.tex_bits = nullptr; tb.tex_odd = nullptr; tb.sector_cached = 0; tb.tex_cached = 0;
    const int y = pixel / SW, x = pixel - y * SW;
    const size_t i = (size_t)local * VH * SW + pixel;
    const int s = sc.flat_sector[i];
    const float delta = (float)y - flat_center(c);
    frame[pixel] = flat_pixel(tb, m->colormap, c, s, delta > 0, x, y);
}

__global__ void __launch_bounds__(64) flat_shade_kernel(DeviceMap dm, Scratch sc, unsigned char *frame_base, size_t frame_stride) {
    const int total = *sc.gap_column_count;
    for (int entry = blockIdx.x; entry < total; entry += gridDim.x) {
        const int2 packed = sc.gap_columns[entry];
        const int local = packed.x >> 9, x = packed.x & 511, last = packed.y >> 8;
        for (int y = (packed.y & 255) + (int)threadIdx.x; y < last; y += 64) {
            const unsigned int word = sc.meta[(size_t)local * VH * SW + (size_t)y * SW + x];
            if (gap_pixel(word) && !(word & META_GAP_COVERED))
                flat_shade_pixel(dm, sc, sc.ctx[local], local, y * SW + x, frame_base + (size_t)local * frame_stride);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// sprites: engine.py:10534-10557 (blocking raycast) and 14684-14947
// ---------------------------------------------------------------------------------------------
#define SPRITE_ROWS 4   // rows of a sprite column in flight together (sprite_column)
// One billboard seen from one lane.  Pixels of a wavefront read different records of an LDS array: 104 bytes, 26 words,
// spread them over the banks (96 would put every eighth record on the same one).
struct SpriteRec {
    float x, y, depth;
    int height;
    i64 depth_fixed, left, right, hstep, yscale, top_fixed, fraction_base, iscale;
    size_t texel_base;   // first texel of the patch in the atlas
    int slot, flags;   // bits 0..4 colormap row, bits 8..15 style (signed: -1 opaque, -2 translucent, >= 0 additive),
                       // bits 16..23 / 24..31 first / one past the last screen row the patch can reach
    int width, spare;
};
static_assert(sizeof(SpriteRec) == 104, "SpriteRec: 26 words");

// Slot `a` of lane `n` as a record (engine.py:14684-14760); false if it cannot reach columns [x_first, x_end) and rows
// [row_first, row_end) at all (dead, not in front, none of its columns or rows in them).
__device__ __forceinline__ bool sprite_record(const DeviceMap &dm, const gd_lanes_desc &lanes, int n, const LaneCtx &L, int a, int x_first, int x_end,
                                              int row_first, int row_end, SpriteRec &s) {
    const gd_map_desc *m = &dm.d;
    const size_t k = (size_t)n * lanes.sprite_slots + a;
    const int id = lanes.sprite_id[k];
    s.depth = lanes.sprite_depth[k];
    if (!lanes.sprite_alive[k] || id < 0 || id >= m->sprite_count || !(s.depth > 0)) return false;   // an unknown patch id is never drawn
    s.x = lanes.sprite_x[k]; s.y = lanes.sprite_y[k];
    const float z = lanes.sprite_z[k];
    const i64 ax = round_to_i64(s.x * 65536.0f), ay = round_to_i64(s.y * 65536.0f);
    const i64 rx = ax - L.view_x_fixed, ry = ay - L.view_y_fixed;
    s.depth_fixed = (rx * L.vcos + ry * L.vsin) >> 20;
    const i64 side_fixed = (rx * L.vsin - ry * L.vcos) >> 16;
    const i64 xscale = tdiv(FOCAL_X_FIXED << 12, max64(s.depth_fixed, SPRITE_MIN_DEPTH_FIXED));
    const i64 left_fixed = side_fixed - (i64)m->spr_left[id] * FIXED_UNIT;
    s.width = m->spr_w[id];
    s.left = SW / 2 + (mul64(left_fixed, xscale) >> 32);
    const i64 right_fixed = left_fixed + (i64)s.width * FIXED_UNIT;
    s.right = SW / 2 + (mul64(right_fixed, xscale) >> 32);
    if (!(s.right > x_first && s.left < x_end && s.right > s.left)) return false;
    s.height = m->spr_h[id];
    s.hstep = tdiv((i64)s.width << 16, max64(s.right - s.left, 1));
    s.yscale = tdiv(FOCAL_Y_FIXED << 12, max64(s.depth_fixed, SPRITE_MIN_DEPTH_FIXED));
    const i64 texmid = (i64)m->spr_top[id] * FIXED_UNIT - round_to_i64((L.view_z - z) * 65536.0f);
    s.top_fixed = L.center_fixed - (mul64(texmid, s.yscale) >> 16);
    s.iscale = tdiv(UINT32_MASK, max64(s.yscale, 1));
    // Screen row y shows source row (fraction_base + y * iscale) >> 16 (engine.py:14830-14846).  The rows whose source
    // row can fall inside the patch: a bracket from two divisions, a row too wide on either side; the exact test
    // stays per row.
    s.fraction_base = texmid - (mul64(L.center_fixed - FIXED_UNIT, s.iscale) >> 16);
    int y_lo = 0, y_hi = VH;
    if (s.iscale > 0) {
        y_lo = (int)clampi(tdiv(-s.fraction_base, s.iscale) - 1, 0, VH);
        y_hi = (int)clampi(tdiv(((i64)s.height << 16) - s.fraction_base, s.iscale) + 2, 0, VH);
    }
    if (!(y_hi > row_first && y_lo < row_end)) return false;
    float light = m->sector_lights[sector_at(m, s.x, s.y)] + (float)(L.flash_light * 16);
    if (lanes.sprite_fullbright && lanes.sprite_fullbright[k]) light = 255.0f;
    const float base_shade = 61.0f - light / 4.0f;
    // engine.py:10583 divides a Python number by a tensor, which Torch evaluates as reciprocal(distance) * 1280
    // (Tensor.__rtruediv__): two roundings, not one division
    const float visibility = fminf((1.0f / fmaxf(s.depth, 1.0f)) * 1280.0f, 24.0f);
    const int shade = (int)clampi((i64)floorf(base_shade - visibility), 0, 31);
    const int style = lanes.sprite_style ? (int)lanes.sprite_style[k] : -1;
    s.flags = (int)((unsigned)shade | (((unsigned)style & 0xFFu) << 8) | ((unsigned)y_lo << 16) | ((unsigned)y_hi << 24));
    s.texel_base = (size_t)id * m->spr_max_h * m->spr_max_w;
    s.slot = a; s.spare = 0;
    return true;
}

// A lane's billboards that reach the given part of the view, one record per entry in no particular order (there is room for
// every slot): the loops over billboards only walk these.  `listed` starts at 0.
__device__ __forceinline__ void stage_sprites(const DeviceMap &dm, const gd_lanes_desc &lanes, int n, const LaneCtx &L, int x_first, int x_end,
                                              int row_first, int row_end, SpriteRec *sp, int *listed) {
    for (int a = threadIdx.x; a < lanes.sprite_slots; a += blockDim.x) {
        SpriteRec s;
        if (sprite_record(dm, lanes, n, L, a, x_first, x_end, row_first, row_end, s)) sp[atomicAdd(listed, 1)] = s;
    }
}

// The nearest blocking linedef of a column (engine.py:10534-10557), gathered by wall_setup_kernel: what hides a billboard there.
struct ColumnBlocker {
    float distance, dx, dy, ox, oy;
    i64 near, far;
    bool owns;
    __device__ __forceinline__ ColumnBlocker(const DeviceMap &dm, const Scratch &sc, int local, int x) {
        const gd_map_desc *m = &dm.d;
        const u64 hit = sc.block_hit[(size_t)local * SW + x];
        const float best = hit == ~0ULL ? GD_INF : __uint_as_float((unsigned)(hit >> 32));
        const int slot = finitef(best) ? (int)(hit & 0xFFFFFFFFu) : 0;
        distance = fminf(fmaxf(best, 1.0f), 4096.0f);
        const int bw = m->blocking_count ? m->blocking_walls[slot] : 0;
        const WallRec &bg = sc.rec[(size_t)local * m->wall_count + bw];
        near = min64(bg.dl, bg.dr); far = max64(bg.dl, bg.dr);
        const float4 bl = *reinterpret_cast<const float4 *>(m->walls + 4 * bw);
        dx = bl.z - bl.x; dy = bl.w - bl.y; ox = bl.x; oy = bl.y;
        owns = (x >= bg.sl) && (x < bg.sr);
    }
    // Does billboard `s` cover the column, in front of the blocking linedef?  engine.py:14762-14800
    __device__ __forceinline__ bool shows(const SpriteRec &s, int x) const {
        if (!((x >= s.left) && (x < s.right))) return false;
        bool ray_visible = s.depth < distance;
        if (!ray_visible) {
            const float side = dx * (s.y - oy) - dy * (s.x - ox);
            const bool behind = (near > s.depth_fixed) || ((far > s.depth_fixed) && (side <= 0));
            ray_visible = !owns || behind;
        }
        const i64 su = mul64((i64)x - s.left, s.hstep) >> 16;
        return ray_visible && su >= 0 && su < s.width;
    }
};

// What clips billboards at one view pixel: the linedef of its word or, where there is none but a plane of the wall pass shows, the
// plane's own depth, unless the flat ray resolves there (engine.py:13417-13422).
struct PixelClip {
    i64 near, far;
    float4 line;
    float plane_depth;   // infinite without a plane
    int plane;
    bool by_linedef;
    __device__ __forceinline__ void set(const DeviceMap &dm, const Scratch &sc, int local, const LaneCtx &L, unsigned int word, int y) {
        const gd_map_desc *m = &dm.d;
        const int cw = (int)(word & META_WALL_MASK) - 1;
        by_linedef = cw >= 0;
        plane = -1; plane_depth = GD_INF;
        if (by_linedef) {
            const WallRec &cg = sc.rec[(size_t)local * m->wall_count + cw];
            near = min64(cg.dl, cg.dr); far = max64(cg.dl, cg.dr);
            line = *reinterpret_cast<const float4 *>(m->walls + 4 * cw);
        } else {
            plane = (word & META_FILLED) ? -1 : (int)((word >> META_SECTOR_SHIFT) & META_SECTOR_MASK) - 1;
            if (plane >= 0) {
                const bool plane_floor = (word & META_FLOOR) != 0;
                const float plane_height = plane_floor ? (L.view_z - m->sector_heights[2 * plane]) : (m->sector_heights[2 * plane + 1] - L.view_z);
                plane_depth = plane_height * 192.0f / fmaxf(fabsf((float)y - ((103.0f + L.pitch_offset) + 0.5f)), 0.5f);
            }
        }
    }
    __device__ __forceinline__ bool linedef_shows(const SpriteRec &s) const {
        const float side = (line.z - line.x) * (s.y - line.y) - (line.w - line.y) * (s.x - line.x);
        return (near > s.depth_fixed) || ((far > s.depth_fixed) && (side <= 0));
    }
};

// engine.py:14914-14939: opaque, additive table or translucent table over the pixel below
__device__ __forceinline__ unsigned char sprite_blend(const gd_map_desc *m, int style, unsigned char lit, unsigned char below) {
    if (style == -2) return m->translucent_lut[(size_t)below * 256 + lit];
    if (style >= 0) return m->additive_luts[((size_t)(style > 1 ? 1 : style) * 256 + below) * 256 + lit];
    return lit;
}

__device__ __forceinline__ bool sprite_blends(const SpriteRec &s) { const int style = (int)(signed char)(s.flags >> 8); return style == -2 || style >= 0; }

// Every billboard of column x, rows [row_first, row_end), far -> near (engine.py:14762-14947): band_finish_kernel's way, one thread
// a column and SPRITE_ROWS rows in flight, over a frame whose rows lie in LDS.
template <typename Frame>
__device__ __forceinline__ void sprite_column(const DeviceMap &dm, const gd_lanes_desc &lanes, const Scratch &sc, int local, int n, const LaneCtx &L,
                                              const SpriteRec *sp, int listed, int x, int row_first, int row_end, const Frame &frame) {
    const gd_map_desc *m = &dm.d;
    const unsigned int *meta = sc.meta + (size_t)local * VH * SW;
    const ColumnBlocker blocker(dm, sc, local, x);
    u64 cover[8];   // the billboards of the column, a bit an entry (sprite_slots <= 512)
#pragma unroll
    for (int word = 0; word < 8; ++word) {
        cover[word] = 0;
        if (word * 64 >= listed) continue;     // the same in every thread
        const int end = listed - word * 64 < 64 ? listed - word * 64 : 64;
        for (int b = 0; b < end; ++b) if (blocker.shows(sp[word * 64 + b], x)) cover[word] |= 1ULL << b;
    }
    // painter's order far -> near: repeatedly take the farthest candidate nearer than the last one
    float last_depth = GD_INF; int last_slot = lanes.sprite_slots;
    for (;;) {
        float pick_depth = -GD_INF; int pick = -1, pick_slot = -1;
#pragma unroll
        for (int word = 0; word < 8; ++word) {
            for (u64 bits = cover[word]; bits; bits &= bits - 1) {
                const int at = word * 64 + __ffsll((long long)bits) - 1;
                const float depth = sp[at].depth; const int a = sp[at].slot;
                // strictly before (last_depth, last_slot) in (depth, slot) order
                if (!(depth < last_depth || (depth == last_depth && a < last_slot))) continue;
                if (depth > pick_depth || (depth == pick_depth && a > pick_slot)) { pick_depth = depth; pick = at; pick_slot = a; }
            }
        }
        if (pick < 0) break;
        last_depth = pick_depth; last_slot = pick_slot;
        const SpriteRec &s = sp[pick];
        const i64 su = mul64((i64)x - s.left, s.hstep) >> 16;
        const int style = (int)(signed char)(s.flags >> 8), shade = s.flags & 31;
        const int y_lo = max((int)((unsigned)s.flags >> 16) & 255, row_first), y_hi = min((int)((unsigned)s.flags >> 24), row_end);
        // SPRITE_ROWS rows per step, each stage's loads issued together so that their latencies overlap
        for (int yb = y_lo; yb < y_hi; yb += SPRITE_ROWS) {
            bool live[SPRITE_ROWS]; unsigned int row_meta[SPRITE_ROWS];
            unsigned char opaque[SPRITE_ROWS], post_top[SPRITE_ROWS], texel[SPRITE_ROWS];
#pragma unroll
            for (int j = 0; j < SPRITE_ROWS; ++j) {
                const int y = yb + j;
                const i64 sv = (s.fraction_base + mul64((i64)y, s.iscale)) >> 16;
                live[j] = y < y_hi && sv >= 0 && sv < s.height;
                row_meta[j] = meta[(size_t)(y < VH ? y : VH - 1) * SW + x];
                opaque[j] = 0; post_top[j] = 0; texel[j] = 0;
                if (!live[j]) continue;
                const size_t t = s.texel_base + (size_t)sv * m->spr_max_w + su;
                opaque[j] = m->spr_opaque[t]; post_top[j] = m->spr_post_top[t]; texel[j] = m->spr_atlas[t];
            }
#pragma unroll
            for (int j = 0; j < SPRITE_ROWS; ++j) {
                if (!live[j]) continue;
                PixelClip clip;
                clip.set(dm, sc, local, L, row_meta[j], yb + j);
                if (clip.by_linedef) {
                    live[j] = clip.linedef_shows(s);
                } else {
                    live[j] = s.depth < GD_INF;   // no clip linedef: the clip depth is infinite
                    // only a billboard standing behind the plane needs to know whether the flat ray resolves
                    if (live[j] && clip.plane >= 0 && !(s.depth < clip.plane_depth))
                        live[j] = flat_ray_resolves(dm, sc, local, L, lanes.ray_cos[(size_t)n * SW + x], lanes.ray_sin[(size_t)n * SW + x],
                                                    dm.cosine_correction[x], yb + j, clip.plane);
                }
            }
#pragma unroll
            for (int j = 0; j < SPRITE_ROWS; ++j) {
                if (!live[j] || !opaque[j]) continue;
                const int y = yb + j;
                if ((i64)y < ((s.top_fixed + mul64(s.yscale, post_top[j])) >> 16)) continue;
                unsigned char *pixel = frame.at(y, x);
                *pixel = sprite_blend(m, style, m->colormap[shade * 256 + texel[j]], *pixel);
            }
        }
    }
}

// The billboards of a lane that reach the view, for all the work-groups that paint its columns: their records in no order, and their
// places and reach near to far, equal depths by slot.  They lie where the lane's candidate lists were, which nothing reads once every
// strip is selected.
#define SPRITE_SLOTS_MAX 512
struct __align__(8) SpriteHead {
    short x0, x1;            // columns and rows of the view it can reach
    unsigned char y0, y1;
    unsigned short record;
};
static_assert(SPRITE_SLOTS_MAX * (sizeof(SpriteRec) + sizeof(SpriteHead)) <= CAND_MAX * SW * sizeof(Cand), "sprite lists: room in a lane's candidate lists");
__device__ __forceinline__ SpriteRec *sprite_records(const Scratch &sc, int local) { return reinterpret_cast<SpriteRec *>(sc.cand + (size_t)local * CAND_MAX * SW); }
__device__ __forceinline__ SpriteHead *sprite_heads(const Scratch &sc, int local) { return reinterpret_cast<SpriteHead *>(sprite_records(sc, local) + SPRITE_SLOTS_MAX); }

// One work-group per lane.  It runs beside the drawing of the walls: the work-groups that paint 64 columns each used to work out the records
// of all slots, five times a lane, and to order their own lists, which was what they were bound by.  0.05 ms for 4096 lanes with 128 slots,
// hidden behind wall_geometry_kernel and wall_raster_kernel.
#define LIST_THREADS 128
__global__ void __launch_bounds__(LIST_THREADS) sprite_list_kernel(DeviceMap dm, gd_lanes_desc lanes, int lane_base, int lane_count, Scratch sc) {
    __shared__ float depth_of[SPRITE_SLOTS_MAX];
    __shared__ unsigned short slot_of[SPRITE_SLOTS_MAX];
    __shared__ SpriteHead head_of[SPRITE_SLOTS_MAX];
    __shared__ int listed_count;
    const int local = blockIdx.x;
    if (local >= lane_count) return;
    if (threadIdx.x == 0) listed_count = 0;
    __syncthreads();
    const LaneCtx &L = sc.ctx[local];
    SpriteRec *records = sprite_records(sc, local);
    for (int a = threadIdx.x; a < lanes.sprite_slots; a += LIST_THREADS) {
        SpriteRec s;
        if (!sprite_record(dm, lanes, lane_base + local, L, a, 0, SW, 0, VH, s)) continue;
        const int at = atomicAdd(&listed_count, 1);
        records[at] = s;
        depth_of[at] = s.depth; slot_of[at] = (unsigned short)a;
        SpriteHead h;
        h.x0 = (short)clampi(s.left, 0, SW); h.x1 = (short)clampi(s.right, 0, SW);
        h.y0 = (unsigned char)((unsigned)s.flags >> 16); h.y1 = (unsigned char)((unsigned)s.flags >> 24);
        h.record = (unsigned short)at;
        head_of[at] = h;
    }
    __syncthreads();
    const int listed = listed_count;
    if (threadIdx.x == 0) sc.sprite_listed[local] = listed;
    SpriteHead *heads = sprite_heads(sc, local);
    for (int i = threadIdx.x; i < listed; i += LIST_THREADS) {   // an entry's place is the number of entries before it
        const float depth = depth_of[i]; const int slot = slot_of[i];
        int before = 0;
        for (int j = 0; j < listed; ++j) before += depth_of[j] < depth || (depth_of[j] == depth && slot_of[j] < slot);
        heads[before] = head_of[i];
    }
}

// A thread a view pixel.  A work-group takes SPRITE_COLUMNS columns of a lane and 1 / gridDim.z of its rows: it picks the billboards that
// reach them from the lane's list, near to far, and notes as bit sets over that order which entries show in each
// column and which have a source row in each row; a pixel then walks the entries in both sets and stops at the first that is
// visible and opaque there (in a lane with billboards that blend it then goes back over those it passed).  What clips
// billboards at the pixel is read once, not once per billboard: on the 4000-linedef map most of what a column ray passes is behind
// walls, and a column's thread used to read word, linedef and patch for every row of every one of them (and the flat ray's
// decision, which does not depend on the billboard, each time as well), waiting for one before the next.
// A list longer than SPRITE_CHUNK, one word of bits, is painted in chunks of that many, the farthest first: the LDS a group
// needs does not follow the slots a lane has.
// Bound by the waits of pixels that show something: their clip, their texels (one word: three bytes each cost 3 % more), and the flat ray.
// BLENDS: frames with sprite_style.  The others have no use for what blending takes: five registers of the seven spilled (a frame of 4096 lanes
// 3825 -> 3810 us without).  Five wavefronts a SIMD are better than four by 4 %, six worse by 25 %; four for the early launch that blends, which would
// spill 17 (1024 lanes, a quarter of them blending, 1054 -> 1051 us).
#define SPRITE_THREADS 256
#define SPRITE_TILE_W 16      // columns of a wavefront's tile: 8 to 64 within 3 %
#define SPRITE_TILE_H (64 / SPRITE_TILE_W)
#define SPRITE_TILES 4        // tiles of a wavefront whose words are asked for together
#define SPRITE_CHUNK 64
#define SPRITE_COLUMNS 64     // a work-group for the whole lane: 0.95 ms instead of 0.70 (4 wavefronts), 0.86 (8)
static_assert(SPRITE_COLUMNS == 64 && SW % SPRITE_COLUMNS == 0 && VH % (SPRITE_ROW_PARTS * SPRITE_TILE_H) == 0 && VH <= SPRITE_THREADS, "sprite_pixels_kernel: whole tiles");
static_assert(SPRITE_CHUNK == 64 && SPRITE_CHUNK <= SPRITE_THREADS, "sprite_pixels_kernel: a bit an entry");
template <int PHASE, bool BLENDS>
__global__ void __launch_bounds__(SPRITE_THREADS, PHASE == SPRITES_EARLY && BLENDS ? 4 : 5) sprite_pixels_kernel(DeviceMap dm, gd_lanes_desc lanes, int lane_base, int lane_count, Scratch sc,
                                                                          unsigned char *frame_base, size_t frame_stride) {
    __shared__ SpriteRec sp[SPRITE_CHUNK];         // the chunk's records, near to far
    __shared__ u64 cover[SPRITE_COLUMNS], in_row[VH];
    __shared__ unsigned short picked[SPRITE_SLOTS_MAX];   // the records of the billboards that reach the group's columns and rows, near to far
    __shared__ int wave_picks[SPRITE_SLOTS_MAX / 64], next_tile, left_over;
    const int local = blockIdx.y;
    if (local >= lane_count) return;
    // SPRITES_EARLY: all but gap pixels that show billboards which blend, and none that covers, since what is under them is not painted yet.
    // SPRITES_LATE: those, in the groups that have any.
    const bool blends = BLENDS && sc.lane_blends[local] != 0;
    const auto late = [&]() -> unsigned char & { return sc.sprite_late[((size_t)local * (SW / SPRITE_COLUMNS) + blockIdx.x) * SPRITE_ROW_PARTS + blockIdx.z]; };
    if (PHASE == SPRITES_LATE && (!blends || late() == 0)) return;     // the same in the whole block
    if (PHASE == SPRITES_EARLY && blends && threadIdx.x == 0) { late() = 0; left_over = 0; }
    const gd_map_desc *m = &dm.d;
    const int n = lane_base + local, tid = threadIdx.x;
    const int rows = VH / gridDim.z;
    const int x_first = blockIdx.x * SPRITE_COLUMNS, row_first = blockIdx.z * rows;
    const LaneCtx &L = sc.ctx[local];
    const int lane_id = tid & 63, wave = tid >> 6;
    constexpr int WAVES = SPRITE_THREADS / 64;
    const int on_view = sc.sprite_listed[local];
    if (on_view == 0) return;                      // the same in the whole block
    const SpriteHead *heads = sprite_heads(sc, local);
    u64 picks[SPRITE_SLOTS_MAX / SPRITE_THREADS]; unsigned short record[SPRITE_SLOTS_MAX / SPRITE_THREADS];
#pragma unroll
    for (int k = 0; k < SPRITE_SLOTS_MAX / SPRITE_THREADS; ++k) {   // 64 entries a wavefront and turn
        const int i = k * SPRITE_THREADS + tid;
        picks[k] = 0; record[k] = 0;
        if (k * SPRITE_THREADS >= on_view) continue;                // the same in the whole block
        bool pick = false;
        if (i < on_view) {
            const SpriteHead head = heads[i];
            pick = head.x1 > x_first && head.x0 < x_first + SPRITE_COLUMNS && head.y1 > row_first && head.y0 < row_first + rows;
            record[k] = head.record;
        }
        picks[k] = __ballot(pick);
        if (lane_id == 0) wave_picks[k * WAVES + wave] = __popcll(picks[k]);
    }
    __syncthreads();
    int listed = 0;
#pragma unroll
    for (int k = 0; k < SPRITE_SLOTS_MAX / SPRITE_THREADS; ++k) {
        if (k * SPRITE_THREADS >= on_view) continue;
        int before = listed;
#pragma unroll
        for (int q = 0; q < WAVES; ++q) { before += q < wave ? wave_picks[k * WAVES + q] : 0; listed += wave_picks[k * WAVES + q]; }
        if ((picks[k] >> lane_id) & 1) picked[before + __popcll(picks[k] & ((1ULL << lane_id) - 1))] = record[k];
    }
    if (listed == 0) return;                       // the same in the whole block
    __syncthreads();
    const unsigned int *records = reinterpret_cast<const unsigned int *>(sprite_records(sc, local));
    unsigned int *meta = sc.meta + (size_t)local * VH * SW;
    unsigned char *frame = frame_base + (size_t)local * frame_stride;
    constexpr int TILES_ACROSS = SPRITE_COLUMNS / SPRITE_TILE_W;
    const int tiles = TILES_ACROSS * (rows / SPRITE_TILE_H);
    const int tile_x = lane_id % SPRITE_TILE_W, tile_y = lane_id / SPRITE_TILE_W;
    for (int first = (listed - 1) / SPRITE_CHUNK * SPRITE_CHUNK; first >= 0; first -= SPRITE_CHUNK) {
        const int length = listed - first < SPRITE_CHUNK ? listed - first : SPRITE_CHUNK;
        {   // the chunk's records into their places
            constexpr int WORDS = sizeof(SpriteRec) / 4;
            if (first + SPRITE_CHUNK < listed) __syncthreads();   // every pixel of the chunk before is painted: its records and bit sets are free
            for (int k = tid; k < length * WORDS; k += SPRITE_THREADS) {
                const int entry = k / WORDS;
                reinterpret_cast<unsigned int *>(sp)[k] = records[picked[first + entry] * WORDS + (k - entry * WORDS)];
            }
            if (tid < SPRITE_COLUMNS) cover[tid] = 0;
            if (tid == 0) next_tile = 0;
            __syncthreads();
        }
        {   // a column's entries are shared out over the wavefronts
            const ColumnBlocker blocker(dm, sc, local, x_first + lane_id);
            u64 bits = 0;
            for (int b = wave; b < length; b += WAVES) if (blocker.shows(sp[b], x_first + lane_id)) bits |= 1ULL << b;
            if (bits) atomicOr(&cover[lane_id], bits);
        }
        if (tid < rows) {
            const int y = row_first + tid;
            u64 bits = 0;
            for (int b = 0; b < length; ++b) {
                const SpriteRec &s = sp[b];
                const i64 sv = (s.fraction_base + mul64((i64)y, s.iscale)) >> 16;
                if (y >= (int)(((unsigned)s.flags >> 16) & 255) && y < (int)((unsigned)s.flags >> 24) && sv >= 0 && sv < s.height) bits |= 1ULL << b;
            }
            in_row[tid] = bits;
        }
        __syncthreads();
        // Wavefronts take the next tiles when they are done with theirs: what a tile costs ranges from a look at two bit sets to
        // several rounds of patch texels and the flat ray's decision.
        for (;;) {
            int t0 = 0;
            if (lane_id == 0) t0 = atomicAdd(&next_tile, SPRITE_TILES);
            t0 = __builtin_amdgcn_readfirstlane(t0);
            if (t0 >= tiles) break;
            unsigned int pixel_words[SPRITE_TILES];
            u64 entries[SPRITE_TILES];
#pragma unroll
            for (int j = 0; j < SPRITE_TILES; ++j) {
                const int t = t0 + j;
                entries[j] = 0; pixel_words[j] = 0;
                if (t >= tiles) continue;              // the same in the whole wavefront
                const int column = t % TILES_ACROSS * SPRITE_TILE_W + tile_x, row = t / TILES_ACROSS * SPRITE_TILE_H + tile_y;
                entries[j] = cover[column] & in_row[row];
                if (entries[j]) pixel_words[j] = meta[(size_t)(row_first + row) * SW + x_first + column];
            }
#pragma unroll
            for (int j = 0; j < SPRITE_TILES; ++j) {
                if (!entries[j]) continue;
                const int t = t0 + j;
                const int x = x_first + t % TILES_ACROSS * SPRITE_TILE_W + tile_x, y = row_first + t / TILES_ACROSS * SPRITE_TILE_H + tile_y;
                const unsigned int pixel_word = pixel_words[j];
                const bool open_gap = gap_pixel(pixel_word) && !(pixel_word & META_GAP_COVERED);
                if (PHASE == SPRITES_LATE && !open_gap) continue;
                PixelClip clip;
                clip.set(dm, sc, local, L, pixel_word, y);
                unsigned char *pixel = frame + (size_t)y * SW + x;
                int value = -1;                        // what the pixel shows, once a billboard does
                int resolves = -1;                     // does the flat ray resolve here: not known, no, yes
                // is the billboard in front of what clips it here: no, yes, -1 = ask the flat ray first
                auto in_front = [&](const SpriteRec &s) -> int {
                    if (clip.by_linedef) return clip.linedef_shows(s);
                    if (!(s.depth < GD_INF)) return 0;                                       // no clip linedef: the clip depth is infinite
                    return (clip.plane < 0 || s.depth < clip.plane_depth) ? 1 : resolves;    // only a billboard standing behind the plane needs to know
                };
                // its colour at the pixel after the colormap, -1 where the patch has none
                auto colour = [&](const SpriteRec &s) -> int {
                    const i64 su = mul64((i64)x - s.left, s.hstep) >> 16, sv = (s.fraction_base + mul64((i64)y, s.iscale)) >> 16;
                    const unsigned int texel = dm.sprite_texels[s.texel_base + (size_t)sv * m->spr_max_w + su];
                    if (!(texel >> 16) || (i64)y < ((s.top_fixed + mul64(s.yscale, (texel >> 8) & 255u)) >> 16)) return -1;
                    return m->colormap[(s.flags & 31) * 256 + (texel & 255u)];
                };
                u64 bits = entries[j], blended = 0;
                bool undecided;
                do {
                    undecided = false;
                    while (bits) {
                        const int bit = __ffsll((long long)bits) - 1;
                        const SpriteRec &s = sp[bit];
                        const int front = in_front(s);
                        if (front < 0) { undecided = true; break; }
                        bits &= bits - 1;
                        if (!front) continue;
                        if (blends && sprite_blends(s)) { blended |= 1ULL << bit; continue; }
                        value = colour(s);
                        if (value >= 0) bits = 0;
                    }
                    // a pixel that has to know whether its flat ray resolves leaves the walk for it, once: those that do ask together
                    if (undecided)
                        resolves = flat_ray_resolves(dm, sc, local, L, lanes.ray_cos[(size_t)n * SW + x], lanes.ray_sin[(size_t)n * SW + x],
                                                     dm.cosine_correction[x], y, clip.plane) ? 1 : 0;
                } while (undecided);
                if (blended) {                         // from the opaque entry back to the eye
                    bool below_known = value >= 0;
                    while (blended) {
                        const int bit = 63 - __clzll((long long)blended);
                        blended &= ~(1ULL << bit);
                        const SpriteRec &s = sp[bit];
                        const int lit = colour(s);
                        if (lit < 0) continue;
                        if (!below_known && PHASE == SPRITES_EARLY && open_gap) { left_over = 1; break; }
                        if (!below_known) { value = *pixel; below_known = true; }
                        value = sprite_blend(m, (int)(signed char)(s.flags >> 8), (unsigned char)lit, (unsigned char)value);
                    }
                }
                if (value < 0) continue;
                *pixel = (unsigned char)value;
                // painted ahead of the flat pass's pixels (launch_chunk): a gap pixel says that it is taken
                if (PHASE == SPRITES_EARLY && open_gap) meta[(size_t)y * SW + x] = pixel_word | META_GAP_COVERED;
            }
        }
    }
    if (PHASE != SPRITES_EARLY || !blends) return;
    __syncthreads();
    if (tid == 0 && left_over) late() = 1;
}

// ---------------------------------------------------------------------------------------------
// wall decals: engine.py:13747-13991, drawn after the walls and before the sprites
// ---------------------------------------------------------------------------------------------
// One thread per screen column; a lane's decals are painted oldest first, each only where the scene
// depth is the decal's own ray distance (which ties it to the wall tier it sits on).  What the walls drew has its depth in
// Scratch::scene_depth; that of the other pixels follows from their words, and only the few a decal reaches are asked for it (a plane
// of it, stored by the shading for every plane pixel, made that kernel 0.75 ms instead of 0.57 for 2048 lanes, beside the flat pass).
__device__ __forceinline__ float scene_depth_at(const DeviceMap &dm, const Scratch &sc, const LaneCtx &c, size_t i, int x, int y) {
    const gd_map_desc *m = &dm.d;
    const unsigned int word = sc.meta[i];
    if (word & (META_FILLED | META_MASKED)) return sc.scene_depth[i];
    const int plane = (int)((word >> META_SECTOR_SHIFT) & META_SECTOR_MASK) - 1;
    if (plane >= 0) {   // exact plane depth (engine.py:13406-13416)
        const float plane_height = (word & META_FLOOR) ? (c.view_z - m->sector_heights[2 * plane]) : (m->sector_heights[2 * plane + 1] - c.view_z);
        return plane_height * 192.0f / fmaxf(fabsf((float)y - ((103.0f + c.pitch_offset) + 0.5f)), 0.5f);
    }
    // the depth the flat pass leaves (engine.py:11140-11166)
    const int s = sc.flat_sector[i], flags = sc.flat_flags[i];
    const float delta = (float)y - flat_center(c);
    const float plane_height = delta > 0 ? (c.view_z - m->sector_heights[2 * s]) : (m->sector_heights[2 * s + 1] - c.view_z);
    const float perpendicular = plane_height * 192.0f / fmaxf(fabsf(delta), 0.5f);
    if (flags & (2 | 8)) return perpendicular;             // repaired: its visplane's depth
    if (flags & 1) return GD_INF;                          // no sector found along the ray
    const float cosine = dm.cosine_correction[x];
    return (perpendicular / cosine) * cosine;              // ray distance of the hit, corrected back
}

// What is the same in all of a decal's columns is worked out by a lane of the first wavefront, a chunk's decals at once; the columns then go through
// the few that show.  (Every column worked out every live decal, one after the other: 71 us for 2048 lanes of 64 slots, an eighth of them in
// use; now 40.)
#define DECAL_CHUNK 64
struct DecalRec {
    float left_x, left_y, seg_x, seg_y;      // its left end and the way to its right end
    float impact_z, light;
    int columns;                             // screen columns it can show in: first | one past the last << 16
    int style;                               // variant | mirrored along the linedef << 8 | mirrored in height << 9
};
__global__ void __launch_bounds__(SW) decal_kernel(DeviceMap dm, Overlays ov, gd_lanes_desc lanes, int lane_base, int lane_count, Scratch sc,
                                                   unsigned char *frame_base, size_t frame_stride) {
    __shared__ DecalRec records[DECAL_CHUNK];
    __shared__ int record_count;
    const gd_map_desc *m = &dm.d;
    const gd_overlay_desc &o = ov.d;
    const int local = blockIdx.x;
    if (local >= lane_count) return;
    const int n = lane_base + local;
    const int x = threadIdx.x;
    const LaneCtx &L = sc.ctx[local];
    const int D = lanes.decal_slots;
    const int width = o.decal_max_w;
    const float center = 104.0f + L.pitch_offset;
    unsigned char *frame = frame_base + (size_t)local * frame_stride;
    float rx, ry; ray_direction(L, x, &rx, &ry);
    for (int first = 0; first < D; first += DECAL_CHUNK) {
        __syncthreads();                     // nobody reads the chunk before any more
        if (x < DECAL_CHUNK) {               // the first wavefront: a lane a decal
            DecalRec r = {};
            bool shows = false;
            const int k = first + x;
            if (k < D) {
                const int *state = lanes.decal_state + ((size_t)n * D + k) * 3;
                const float *geom = lanes.decal_geom + ((size_t)n * D + k) * 4;
                const int wall_index = (int)clampi(state[0], 0, m->wall_count - 1);
                const int style = state[1];
                const int variant = style % 5, side = style / 20;
                const float along_wall = geom[0], tangent_x = geom[2], tangent_y = geom[3];
                const float4 wl = *reinterpret_cast<const float4 *>(m->walls + 4 * wall_index);
                const float wvx = wl.z - wl.x, wvy = wl.w - wl.y;
                const float viewer_cross = wvx * (L.y - wl.y) - wvy * (L.x - wl.x);
                shows = state[2] && (viewer_cross > 0 ? 1 : 0) == side;
                if (shows) {
                    const float impact_x = wl.x + along_wall * wvx, impact_y = wl.y + along_wall * wvy;
                    const float left_offset = (float)o.decal_left[variant];
                    const float back = left_offset * 0.5f, forth = ((float)width - left_offset) * 0.5f;
                    const float left_x = impact_x - tangent_x * back, left_y = impact_y - tangent_y * back;
                    const float right_x = impact_x + tangent_x * forth, right_y = impact_y + tangent_y * forth;
                    r.left_x = left_x; r.left_y = left_y; r.seg_x = right_x - left_x; r.seg_y = right_y - left_y;
                    // FWallCoords::Init on the two fixed-point endpoints (engine.py:13836-13887)
                    const i64 lx = round_to_i64(left_x * 65536.0f) - L.view_x_fixed, ly = round_to_i64(left_y * 65536.0f) - L.view_y_fixed;
                    const i64 qx = round_to_i64(right_x * 65536.0f) - L.view_x_fixed, qy = round_to_i64(right_y * 65536.0f) - L.view_y_fixed;
                    const i64 tx1 = (lx * L.vsin - ly * L.vcos) >> 20, ty1 = (lx * L.vcos + ly * L.vsin) >> 20;
                    const i64 tx2 = (qx * L.vsin - qy * L.vcos) >> 20, ty2 = (qx * L.vcos + qy * L.vsin) >> 20;
                    const i64 center_fixed = 160 * FIXED_UNIT;
                    const i64 projected_left = ((center_fixed + tdiv(tx1 * center_fixed, ty1 == 0 ? 1 : ty1)) >> 16) + (tx1 >= 0);
                    const i64 projected_right = ((center_fixed + tdiv(tx2 * center_fixed, ty2 == 0 ? 1 : ty2)) >> 16) + (tx2 >= 0);
                    const i64 left_den = tx1 - tx2 - ty2 + ty1, right_den = ty2 - ty1 - tx2 + tx1;
                    const bool left_inside = (tx1 >= -ty1) && (tx1 <= ty1) && (ty1 != 0);
                    const bool right_inside = (tx2 <= ty2) && (tx2 >= -ty2) && (ty2 != 0);
                    const bool left_clipped = (tx1 < -ty1) && (tx2 >= -ty2) && (left_den != 0);
                    const bool right_clipped = (tx2 > ty2) && (tx1 <= ty1) && (right_den != 0);
                    const i64 screen_left = left_inside ? clampi(projected_left, 0, SW) : 0;
                    const i64 screen_right = right_inside ? clampi(projected_right, 0, SW) : SW;
                    shows = (left_inside || left_clipped) && (right_inside || right_clipped) && (screen_right > screen_left);
                    r.columns = (int)screen_left | ((int)screen_right << 16);
                    r.impact_z = geom[1];
                    int sector = m->wall_sectors[2 * wall_index + (side > 1 ? 1 : side)];
                    if (sector < 0) sector = 0;
                    const bool horizontal = fabsf(wvy) < 1e-6f, vertical = fabsf(wvx) < 1e-6f;
                    r.light = m->sector_lights[sector] + (vertical ? 16.0f : (horizontal ? -16.0f : 0.0f));
                    r.light = r.light + (float)(L.flash_light * 16);
                    r.style = variant | ((style / 5) % 2 ? 1 << 8 : 0) | ((style / 10) % 2 ? 1 << 9 : 0);
                }
            }
            const u64 shown = __ballot(shows);
            if (shows) records[__popcll(shown & ((1ULL << x) - 1))] = r;      // in slot order
            if (x == 0) record_count = __popcll(shown);
        }
        __syncthreads();
        for (int k = 0; k < record_count; ++k) {
            const DecalRec r = records[k];
            if (!(x >= (r.columns & 0xFFFF) && x < (r.columns >> 16))) continue;
            const float off_x = r.left_x - L.x, off_y = r.left_y - L.y;
            const float den = rx * r.seg_y - ry * r.seg_x;
            if (!(fabsf(den) >= 1e-6f)) continue;
            const float distance = (off_x * r.seg_y - off_y * r.seg_x) / den;
            const float decal_along = (off_x * ry - off_y * rx) / den;
            if (!(distance > 0)) continue;
            const int variant = r.style & 255;
            i64 tu = clampi((i64)floorf(decal_along * (float)width), 0, width - 1);
            if (r.style & (1 << 8)) tu = width - 1 - tu;
            const float safe_distance = fmaxf(distance, 1e-6f);
            // engine.py:13909 divides a Python number by a tensor: reciprocal(distance) * 96 in Torch (Tensor.__rtruediv__)
            const float vertical_scale = (1.0f / safe_distance) * 96.0f;
            const float top = center - ((r.impact_z + (float)o.decal_top[variant] * 0.5f) - L.view_z) * 192.0f / safe_distance;
            const i64 depth_fixed = round_to_i64(safe_distance * 4096.0f);
            const i64 shade = wall_shade(r.light, tdiv(WALL_VISIBILITY_FIXED << 12, max64(depth_fixed, 1)));
            const int height = o.decal_h[variant];
            // rows whose source row floor((y - top) / vertical_scale) can fall inside the patch, a row wider
            // on either side; the exact test stays per row
            int y_lo = (int)fminf(fmaxf(floorf(top) - 1.0f, 0.0f), (float)VH);
            int y_hi = (int)fminf(fmaxf(ceilf(top + (float)height * vertical_scale) + 2.0f, 0.0f), (float)VH);
            for (int y = y_lo; y < y_hi; ++y) {
                i64 tv = (i64)floorf(((float)y - top) / vertical_scale);
                if (!(tv >= 0 && tv < height)) continue;
                if (r.style & (1 << 9)) tv = height - 1 - tv;
                const size_t i = (size_t)y * SW + x;
                if (!(fabsf(scene_depth_at(dm, sc, L, (size_t)local * VH * SW + i, x, y) - distance) <= 1e-3f)) continue;
                const unsigned char source = o.decal_atlas[((size_t)variant * o.decal_max_h + tv) * o.decal_max_w + tu];
                if (source == 0) continue;
                const unsigned char opacity = o.decal_opacity_lut[shade * 256 + source];
                frame[i] = o.decal_black_lut[(size_t)opacity * 256 + frame[i]];
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// overlay layers drawn after the sprites
// ---------------------------------------------------------------------------------------------
// One psprite patch as a lane shows it (engine.py:14997-15049, _triton_kernels.py:2611-2634): where its texels lie on the screen.
struct Psprite {
    int left, width, height;      // screen column of its first texel column; the texels there are (0 x 0: no patch)
    i64 row_base;                 // screen row y shows texel row (row_base + y * ROW_STEP) >> 16
    size_t texels;
    // BASEYCENTER 100, weapon top 32 + 0x6000/65536, reciprocal of the 240/200 vertical scale
    static constexpr i64 ROW_STEP = UINT32_MASK / (((i64)GD_SCREEN_HEIGHT * FIXED_UNIT) / 200);
    __device__ __forceinline__ Psprite(const gd_overlay_desc &o, i64 patch, i64 horizontal_fixed, i64 vertical_fixed) {
        left = 0; width = 0; height = 0; row_base = 0; texels = 0;
        if (patch < 0 || patch >= o.weapon_patch_count) return;
        const i64 far = 1LL << 28;            // beyond every screen and patch: a position out there stays out there
        left = (int)clampi((horizontal_fixed - (i64)o.weapon_left[patch] * FIXED_UNIT) >> 16, -far, far);
        width = max(min(o.weapon_w[patch], o.weapon_max_w), 0); height = max(min(o.weapon_h[patch], o.weapon_max_h), 0);   // sizes beyond the atlas: malformed patch
        const i64 texture_mid = 100 * FIXED_UNIT - (32 * FIXED_UNIT + 0x6000) - vertical_fixed + (i64)o.weapon_top[patch] * FIXED_UNIT;
        row_base = clampi(texture_mid, -(far << 16), far << 16) - (VH / 2 - 1) * ROW_STEP;
        texels = (size_t)patch * o.weapon_max_h * o.weapon_max_w;
    }
    // The rectangle of the view outside which the patch has no texel: exact columns, the rows one too many at most on either side.
    __device__ __forceinline__ void bounds(int &x0, int &y0, int &x1, int &y1) const {
        if (width == 0 || height == 0) return;
        x0 = min(x0, max(left, 0)); x1 = max(x1, min(left + width, SW));
        y0 = min(y0, (int)clampi(-row_base / ROW_STEP - 1, 0, VH)); y1 = max(y1, (int)clampi((((i64)height << 16) - row_base) / ROW_STEP + 2, 0, VH));
    }
    __device__ __forceinline__ bool texel(const gd_overlay_desc &o, int px, int py, unsigned char *value) const {
        const int x = px - left;
        const i64 y = (row_base + py * ROW_STEP) >> 16;
        if (x < 0 || x >= width || y < 0 || y >= height) return false;
        const size_t t = texels + (size_t)y * o.weapon_max_w + (size_t)x;
        *value = o.weapon_atlas[t];                // asked for along with the mask, whatever that says
        return o.weapon_opaque[t] != 0;
    }
    // The pixel after the weapon patch and its muzzle flash on top of it.
    static __device__ __forceinline__ void paint(const gd_overlay_desc &o, const Psprite &weapon, const Psprite &flash, int px, int py, unsigned char *pixel) {
        unsigned char under = 0, over = 0;
        const bool weapon_there = weapon.texel(o, px, py, &under), flash_there = flash.texel(o, px, py, &over);
        if (weapon_there || flash_there) *pixel = flash_there ? over : under;
    }
};

// _native_render_weapon (engine.py:15051-15110): the weapon patch, then its muzzle flash on top.  A work-group goes over its share of
// the rectangle that holds both, a wavefront a row at a time: a thread for every pixel of the view spent its time finding out that
// the patch, a tenth of the view, lies elsewhere.  2048 lanes: 0.271 ms a thread a pixel, 0.050 now (bytes one by one: some 8,400 pixels a lane, four loads each).
#define WEAPON_THREADS 256
#define WEAPON_PARTS 8        // work-groups a lane
__global__ void __launch_bounds__(WEAPON_THREADS) weapon_overlay_kernel(Overlays ov, const int64_t *weapon_state, int lane_base, int lane_count,
                                                                        unsigned char *frame_base, size_t frame_stride) {
    const int local = blockIdx.y;
    if (local >= lane_count) return;
    const int64_t *state = weapon_state + (size_t)(lane_base + local) * 5;
    if (state[4] == 0) return;                    // player dead: no psprite
    const Psprite weapon(ov.d, state[0], state[2], state[3]), flash(ov.d, state[1], state[2], state[3]);
    int x0 = SW, y0 = VH, x1 = 0, y1 = 0;
    weapon.bounds(x0, y0, x1, y1); flash.bounds(x0, y0, x1, y1);
    unsigned char *frame = frame_base + (size_t)local * frame_stride;
    const int lane_id = threadIdx.x & 63, wave = blockIdx.x * (WEAPON_THREADS / 64) + (threadIdx.x >> 6);
    for (int py = y0 + wave; py < y1; py += WEAPON_PARTS * (WEAPON_THREADS / 64)) {
        for (int px = x0 + lane_id; px < x1; px += 64) Psprite::paint(ov.d, weapon, flash, px, py, frame + py * SW + px);
    }
}

// _native_render_hud (engine.py:15153-15267): the status bar is a short list of patches drawn in order, later ones over earlier ones.
#define HUD_ROWS (GD_SCREEN_HEIGHT - VH)
#define HUD_TILE_ROWS 8          // a wavefront's tile: 64 columns of so many rows
#define HUD_TILES ((SW / 64) * (HUD_ROWS / HUD_TILE_ROWS))
#define HUD_ENTRIES 44           // two backgrounds, three large numbers of three digits, two signs, the face, six arms, eight small numbers
struct HudEntry {
    int x0, x1, y0, y1;          // the part of the bar (row 208 is row 0) that the patch covers
    i64 texels;                  // pixel (x, y) shows texel texels + y * hud_max_w + x of the atlas
};

// Entry `k` of the list, each by a lane of its own: the digits of the numbers have places whether there are so many or not.
__device__ __forceinline__ HudEntry hud_entry(const gd_overlay_desc &o, const int *state, int k) {
    int patch = -1, x = 0, y = 0, number = 0, place = -1, right = 0;
    bool small = false;
    if (k < 2) { patch = k; x = k == 0 ? 0 : 104; }
    else if (k < 5) { number = state[0]; place = k - 2; right = 44; y = 3; }
    else if (k < 8) { number = state[1]; place = k - 5; right = 90; y = 3; }
    else if (k == 8) { patch = 12; x = 90; y = 3; }
    else if (k < 12) { number = state[2]; place = k - 9; right = 221; y = 3; }
    else if (k == 12) { patch = 12; x = 221; y = 3; }
    else if (k == 13) { patch = state[3]; x = 143; }
    else if (k < 20) {
        const int arm = k - 14;
        patch = arm < 5 && ((state[4] >> arm) & 1) ? 30 + arm : 38 + arm;
        x = 111 + 12 * (arm % 3); y = arm < 3 ? 4 : 14;
    } else if (k < HUD_ENTRIES) {
        const int row = (k - 20) / 6, which = (k - 20) % 6;
        number = which < 3 ? state[5 + row] : (row == 0 ? 200 : (row == 3 ? 300 : 50));
        place = which % 3; right = which < 3 ? 288 : 314; y = 5 + row * 6; small = true;
    }
    bool glyph = false;
    if (place >= 0) {            // _native_draw_hud_number (engine.py:15186-15207); a sign takes a cell and draws nothing
        const int magnitude = min(abs(max(number, -99)), 999), length = magnitude >= 100 ? 3 : (magnitude >= 10 ? 2 : 1);
        const int digit = place == length - 1 ? magnitude % 10 : (place == length - 2 ? (magnitude / 10) % 10 : magnitude / 100);
        if (place < length) { patch = (small ? 28 : 2) + digit; x = right - (length - place) * (small ? 4 : 14); glyph = true; }
    }
    HudEntry e = {0, 0, 0, 0, 0};
    if (patch < 0 || patch >= o.hud_patch_count) return e;
    // _native_draw_hud_patch (engine.py:15153-15184): position less the patch's own offsets, clipped; a glyph's offsets count twice, as in the reference
    const i64 left = (i64)x - (i64)o.hud_left[patch] * (glyph ? 2 : 1), top = (i64)y - (i64)o.hud_top[patch] * (glyph ? 2 : 1);
    e.x0 = (int)clampi(left, 0, SW); e.x1 = (int)clampi(left + min(o.hud_w[patch], o.hud_max_w), 0, SW);
    e.y0 = (int)clampi(top, 0, HUD_ROWS); e.y1 = (int)clampi(top + min(o.hud_h[patch], o.hud_max_h), 0, HUD_ROWS);
    e.texels = ((i64)patch * o.hud_max_h - top) * o.hud_max_w - left;
    return e;
}

// A wavefront's tile of the bar, a column a lane: each pixel the last listed patch with an opaque texel there.  The lanes hold the list, an entry
// each, and the wavefront goes through the entries that meet its tile, from the last on, until every pixel has its texel: two or three.
// (One thread wrote the list and every pixel walked all of it through the patches' tables: 0.42 ms at 16 lanes, now 18 us; 2048 lanes
// 0.72 and 0.10 ms.  Tiles of 16 or 32 rows: 0.12, 0.11 ms, 28 and 57 us at 16 lanes.)
template <class Put>
__device__ __forceinline__ void hud_tile(const gd_overlay_desc &o, const int *state, int tile, Put put) {
    const int lane_id = threadIdx.x & 63, column = tile % (SW / 64) * 64, x = column + lane_id, y = tile / (SW / 64) * HUD_TILE_ROWS;
    const HudEntry mine = hud_entry(o, state, lane_id);
    u64 entries = __ballot(mine.x0 < column + 64 && mine.x1 > column && mine.y0 < y + HUD_TILE_ROWS && mine.y1 > y);
    unsigned char value[HUD_TILE_ROWS];
    unsigned missing = (1u << HUD_TILE_ROWS) - 1u;
#pragma unroll
    for (int r = 0; r < HUD_TILE_ROWS; ++r) value[r] = 0;
    while (entries != 0 && __ballot(missing != 0u) != 0) {
        const int k = 63 - __clzll((long long)entries);
        entries &= ~(1ULL << k);
        const int x0 = __builtin_amdgcn_readlane(mine.x0, k), x1 = __builtin_amdgcn_readlane(mine.x1, k);
        const int y0 = __builtin_amdgcn_readlane(mine.y0, k), y1 = __builtin_amdgcn_readlane(mine.y1, k);
        const i64 texels = (i64)(((u64)(unsigned)__builtin_amdgcn_readlane((int)(mine.texels >> 32), k) << 32) | (unsigned)__builtin_amdgcn_readlane((int)mine.texels, k));
        unsigned char opaque[HUD_TILE_ROWS], texel[HUD_TILE_ROWS];
#pragma unroll
        for (int r = 0; r < HUD_TILE_ROWS; ++r) {
            opaque[r] = 0; texel[r] = 0;
            if (!((missing >> r) & 1u) || x < x0 || x >= x1 || y + r < y0 || y + r >= y1) continue;
            const size_t t = (size_t)(texels + (i64)(y + r) * o.hud_max_w + x);
            opaque[r] = o.hud_opaque[t]; texel[r] = o.hud_atlas[t];
        }
#pragma unroll
        for (int r = 0; r < HUD_TILE_ROWS; ++r) if (opaque[r]) { value[r] = texel[r]; missing &= ~(1u << r); }
    }
#pragma unroll
    for (int r = 0; r < HUD_TILE_ROWS; ++r) put(x, y + r, value[r]);
}

// A wavefront a tile.
#define HUD_THREADS 256
static_assert(HUD_TILES % (HUD_THREADS / 64) == 0 && HUD_ROWS % HUD_TILE_ROWS == 0, "hud_kernel: whole tiles");
__global__ void __launch_bounds__(HUD_THREADS) hud_kernel(Overlays ov, const int *hud_state, int lane_base, int lane_count, unsigned char *frame_base, size_t frame_stride) {
    const int local = blockIdx.y;
    if (local >= lane_count) return;
    unsigned char *bar = frame_base + (size_t)local * frame_stride + (size_t)VH * SW;
    hud_tile(ov.d, hud_state + (size_t)(lane_base + local) * 9, blockIdx.x * (HUD_THREADS / 64) + (threadIdx.x >> 6),
             [&](int x, int y, unsigned char value) { bar[y * SW + x] = value; });
}

// ---------------------------------------------------------------------------------------------
// observation: _triton_kernels.py:120-177 + engine.py:9545-9548 / 2443-2450
// ---------------------------------------------------------------------------------------------
// One PLAYPAL channel after the pickup (gold) and damage (red) screen blends, evaluated in float32 one
// operation at a time and truncated to a byte (engine.py:15385-15397).
__device__ __forceinline__ unsigned char blended_channel(unsigned char value, int channel, float bonus, float flash) {
    const float gold = channel == 0 ? 215.0f : (channel == 1 ? 186.0f : 69.0f);
    const float red = channel == 0 ? 255.0f : 0.0f;
    float v = (float)value * (1.0f - bonus) + gold * bonus;
    v = v * (1.0f - flash) + red * flash;
    return (unsigned char)fminf(fmaxf(v, 0.0f), 255.0f);
}

// The frame stack of one lane, four pixels (one word per stacked observation) at a time: what the stack holds after
// this call goes to `stack` (when it changes) and to the caller's copy, which is laid out either like the stack
// ([4][84][84]) or with the four stacked values of a pixel next to each other ([84][84][4]).
// `kept` holds the stack's words as they were (unused for a lane that resets).  env.py:678-688, engine.py:15447-15450
__device__ __forceinline__ void store_stack_word(unsigned char *stack_lane, unsigned char *copy_lane, bool copy_hwc, bool aligned, size_t word,
                                                 const unsigned int (&kept)[GD_FRAME_STACK], unsigned int grays, bool resets, int stack_mode) {
    const size_t plane = (size_t)GD_OBS_SIZE * GD_OBS_SIZE;   // bytes per stacked observation
    auto store = [&](unsigned char *p, unsigned int v) {
        if (aligned) *reinterpret_cast<unsigned int *>(p) = v;
        else for (int k = 0; k < 4; ++k) p[k] = (unsigned char)(v >> (8 * k));
    };
    const bool steps = !resets && stack_mode == GD_STACK_STEP;
    unsigned int next[GD_FRAME_STACK];
#pragma unroll
    for (int k = 0; k < GD_FRAME_STACK; ++k) next[k] = resets ? grays : (steps ? (k + 1 < GD_FRAME_STACK ? kept[k + 1] : grays) : kept[k]);
    if (resets || steps) {
#pragma unroll
        for (int k = 0; k < GD_FRAME_STACK; ++k) store(stack_lane + k * plane + word * 4, next[k]);
    }
    if (!copy_lane) return;
    if (!copy_hwc) {
#pragma unroll
        for (int k = 0; k < GD_FRAME_STACK; ++k) store(copy_lane + k * plane + word * 4, next[k]);
        return;
    }
    static_assert(GD_FRAME_STACK == 4, "the interleaved copy packs the four stacked values of a pixel into one word");
#pragma unroll
    for (int j = 0; j < 4; ++j) {   // pixel j of the word
        const unsigned int v = ((next[0] >> (8 * j)) & 255u) | (((next[1] >> (8 * j)) & 255u) << 8) |
                               (((next[2] >> (8 * j)) & 255u) << 16) | (((next[3] >> (8 * j)) & 255u) << 24);
        store(copy_lane + (word * 4 + j) * GD_FRAME_STACK, v);
    }
}

// The pooling of a frame as two products of small whole numbers, which the matrix cores take (v_mfma_i32_16x16x64_i8).  An observation pixel
// covers 240/84 frame rows and 320/84 frame columns; its weights (y_overlap * x_overlap) // 48 are exactly (y_overlap / 12) * (x_overlap / 4),
// since row overlaps are multiples of 12 and column overlaps multiples of 4 (84 = 12 * 7 = 4 * 21, 240 = 12 * 20, 320 = 4 * 80): the
// weighted sum is (down weights) x (colours) x (along weights), both weights banded and below 22.
//   along: a wavefront takes 14 observation columns, whose frame columns lie in a window of 64 that starts on 16 bytes: one product for 16
//     frame rows and a channel.  A lane loads sixteen neighbouring pixels of a row, which is the product's layout.
//   down: 14 observation rows pool exactly 40 frame rows, which lie in three of the tiles of 16 rows of a block of 80.  The sums of the first
//     product stay in the lane that they come out in: the order of a product's inner index is free, and the down weights are laid out
//     in the order that the first product leaves (row 16 t + 4 g + r in byte 4 t + r of the lanes of group g).
// Colours are taken less 128, so that they and the sums' two bytes (256 * high + low, low from -128 to 127) are signed bytes.
// What is left for the vector units is to fetch a pixel's colour and to put the channels in words of their own, some five instructions
// a pixel where sums by multiply-add took 21.  The fetches are from 32 copies of the palette, a bank of LDS each: no two lanes of a half
// wavefront ever meet in a bank.  4096 frames of 240 rows: 0.153 ms by multiply-add, 0.105 ms now (the copy of as many bytes takes 0.066).  Tried:
// colour words as the product's bytes as they are (a quarter of the products, 84 a block instead of 27: 0.145); copies 256 bytes apart, so
// that one byte move makes an address (64 KB a work-group leave one a compute unit: 0.136); all of a block's pixels asked for at once (0.118).
#define OBS_TILE 14             // observation columns of a wavefront, observation rows of a product down the columns
#define OBS_WAVES (GD_OBS_SIZE / OBS_TILE)
#define OBS_THREADS (64 * OBS_WAVES)
#define OBS_BLOCK_ROWS (2 * OBS_TILE)
#define OBS_SOURCE_ROWS (OBS_BLOCK_ROWS * GD_SCREEN_HEIGHT / GD_OBS_SIZE)
#define OBS_BLOCKS (GD_OBS_SIZE / OBS_BLOCK_ROWS)      // a frame's blocks of rows
#define OBS_ROW_TILES (OBS_SOURCE_ROWS / 16)
#define OBS_COPIES 32
#define OBS_AHEAD 2             // tiles whose pixels are asked for ahead
static_assert(OBS_WAVES * OBS_TILE == GD_OBS_SIZE && OBS_BLOCKS * OBS_BLOCK_ROWS == GD_OBS_SIZE, "observe_kernel: whole tiles");
static_assert(OBS_SOURCE_ROWS * GD_OBS_SIZE == OBS_BLOCK_ROWS * GD_SCREEN_HEIGHT && OBS_ROW_TILES * 16 == OBS_SOURCE_ROWS && VH % 16 == 0, "observe_kernel: whole rows");
typedef int int4v __attribute__((ext_vector_type(4)));

struct PoolWeights { unsigned char along[OBS_WAVES][64][16], down[2][64][16]; };   // as the products take them: [tile][lane][byte]
constexpr int obs_window(int tile) {   // the first frame column of a tile's window
    const int first = tile * OBS_TILE * 320 / GD_OBS_SIZE / 16 * 16;
    return first > SW - 64 ? SW - 64 : first;
}
constexpr int overlap(int a0, int a1, int b0, int b1) {
    const int low = a0 > b0 ? a0 : b0, high = a1 < b1 ? a1 : b1;
    return high > low ? high - low : 0;
}
constexpr PoolWeights pool_weights() {
    PoolWeights w{};
    for (int lane = 0; lane < 64; ++lane) {
        const int column = lane & 15, group = lane >> 4;
        for (int k = 0; k < 16 && column < OBS_TILE; ++k) {
            for (int tile = 0; tile < OBS_WAVES; ++tile) {
                const int ox = tile * OBS_TILE + column, x = obs_window(tile) + 16 * group + k;
                w.along[tile][lane][k] = (unsigned char)(overlap(ox * 320, ox * 320 + 320, x * 84, x * 84 + 84) / 4);
            }
            for (int half = 0; half < 2 && k < 12; ++half) {
                const int oy = half * OBS_TILE + column, y = 16 * (2 * half + (k >> 2)) + 4 * group + (k & 3);
                w.down[half][lane][k] = (unsigned char)(overlap(oy * 240, oy * 240 + 240, y * 84, y * 84 + 84) / 12);
            }
        }
    }
    return w;
}
constexpr bool pool_weights_whole() {   // every observation pixel has all its weight: 80 along a row, 20 down a column
    const PoolWeights w = pool_weights();
    for (int column = 0; column < OBS_TILE; ++column) {
        for (int tile = 0; tile < OBS_WAVES; ++tile) {
            int sum = 0;
            for (int k = 0; k < 64; ++k) sum += w.along[tile][column + 16 * (k >> 4)][k & 15];
            if (sum != 80) return false;
        }
        for (int half = 0; half < 2; ++half) {
            int sum = 0;
            for (int k = 0; k < 64; ++k) sum += w.down[half][column + 16 * (k >> 4)][k & 15];
            if (sum != 20) return false;
        }
    }
    return true;
}
static_assert(pool_weights_whole(), "observe_kernel: a tile's window holds its columns, a block's tiles its rows");
__device__ const __align__(16) PoolWeights POOL_WEIGHTS = pool_weights();

// A work-group takes a run of the frames' blocks of rows, a wavefront OBS_TILE observation columns of each.  The next block's pixels are asked
// for as soon as a tile's own are used up.
// ALIGNED: the frames start on 16 bytes.
// FEW: a work-group takes half a block, the rows of one product down the columns (the three tiles that they lie in), and no more: twice the
// work-groups, each with less to do one after the other, which asks for all it reads up front and looks colours up in the palette itself.
// Few frames last as long as one work-group: 1 frame 5.4 us by blocks, 4.6 so; 16 frames 6.2, 4.7 (121 registers, four wavefronts a SIMD).
template <bool ALIGNED, bool FEW>
__global__ void __launch_bounds__(OBS_THREADS, FEW ? 3 : 6) observe_kernel(const unsigned char *indexed, size_t lane_stride, int source_rows, const unsigned char *playpal,
                               int lane_count, unsigned char *obs, unsigned char *frames, const unsigned char *reset_mask, int stack_mode,
                               unsigned char *final_frames, bool final_hwc, const float *blend) {
    __shared__ unsigned int pal[256];   // PLAYPAL after the lane's screen blend, one word per colour (red | green << 8 | blue << 16, each less 128)
    constexpr int COPIES = FEW ? 1 : OBS_COPIES, TILES = FEW ? 3 : OBS_ROW_TILES, AHEAD = FEW ? TILES : OBS_AHEAD;
    constexpr int ROWS = FEW ? OBS_TILE : OBS_BLOCK_ROWS, PARTS = GD_OBS_SIZE / ROWS;      // observation rows of a task, tasks of a frame
    __shared__ __align__(16) unsigned int copies[FEW ? 4 : 256 * OBS_COPIES];
    __shared__ unsigned int gray_words[2][ROWS * GD_OBS_SIZE / 4];
    const int tasks = lane_count * PARTS;
    const int first_task = (int)((long long)tasks * blockIdx.x / gridDim.x), end_task = (int)((long long)tasks * (blockIdx.x + 1) / gridDim.x);
    const int wave = threadIdx.x >> 6, lane_id = threadIdx.x & 63, group = lane_id >> 4, column = lane_id & 15;
    const size_t F = (size_t)GD_OBS_SIZE * GD_OBS_SIZE / 4;     // words per observation
    const bool stack_aligned = ((reinterpret_cast<size_t>(frames) | reinterpret_cast<size_t>(final_frames)) & 3) == 0;
    auto load_word = [](const unsigned char *p, bool aligned) -> unsigned int {
        if (aligned) return *reinterpret_cast<const unsigned int *>(p);
        return (unsigned)p[0] | ((unsigned)p[1] << 8) | ((unsigned)p[2] << 16) | ((unsigned)p[3] << 24);
    };
    const unsigned int at = (unsigned)(obs_window(wave) + 16 * group + column * SW);      // lane strides are multiples of 16, like the window's start
    auto tile_row = [](int part, int t) {      // a tile's first row: half a block's tiles are its first three, or its last
        return (FEW ? part >> 1 : part) * OBS_SOURCE_ROWS + 16 * (t + (FEW && (part & 1) ? OBS_ROW_TILES - TILES : 0));
    };
    auto load_tile = [&](int task, int t) -> uint4 {      // a lane's sixteen pixels of a tile; past the source, or the run, those of some row before
        task = min(task, end_task - 1);
        const int n = task / PARTS, row = min(tile_row(task - n * PARTS, t), source_rows - 16);
        const unsigned char *first = indexed + (size_t)n * lane_stride + (size_t)row * SW;
        if (ALIGNED) return *reinterpret_cast<const uint4 *>(first + at);
        const bool aligned = (reinterpret_cast<size_t>(indexed) & 3) == 0;
        return make_uint4(load_word(first + at, aligned), load_word(first + at + 4, aligned), load_word(first + at + 8, aligned), load_word(first + at + 12, aligned));
    };
    uint4 pixels[TILES];
#pragma unroll
    for (int t = 0; t < AHEAD; ++t) pixels[t] = load_tile(first_task, t);
    const int4v along = *reinterpret_cast<const int4v *>(POOL_WEIGHTS.along[wave][lane_id]);
    const int4v down[2] = {*reinterpret_cast<const int4v *>(POOL_WEIGHTS.down[FEW ? first_task & 1 : 0][lane_id]), *reinterpret_cast<const int4v *>(POOL_WEIGHTS.down[1][lane_id])};
    const unsigned int bank = lane_id & (OBS_COPIES - 1);
    auto colour_of = [&](unsigned int word, int k) {
        const unsigned int index = (word >> (8 * k)) & 255u;
        return FEW ? pal[index] : copies[index * COPIES + bank];
    };
    for (int task = first_task; task < end_task; ++task) {
        const int n = task / PARTS, block = task - n * PARTS;
        unsigned int early[FEW ? GD_FRAME_STACK : 1];      // of few, the stack words that the roll keeps, asked for up front: nothing else goes on meanwhile
        if constexpr (FEW) {
            static_assert(ROWS * GD_OBS_SIZE / 4 <= OBS_THREADS, "observe_kernel: a word a thread");
            const bool keeps = threadIdx.x < ROWS * GD_OBS_SIZE / 4 && frames && !(reset_mask && reset_mask[n]);
#pragma unroll
            for (int f = 0; f < GD_FRAME_STACK; ++f)
                early[f] = keeps ? load_word(frames + ((size_t)n * GD_FRAME_STACK * F + f * F + (size_t)block * (ROWS * GD_OBS_SIZE / 4) + threadIdx.x) * 4, stack_aligned) : 0u;
        }
        if (task == first_task || (blend && block == 0)) {      // nobody reads the last lane's copies any more: its last block has been put together
            if (threadIdx.x < 256) {
                const int k = threadIdx.x;
                unsigned int r = playpal[3 * k], g = playpal[3 * k + 1], b = playpal[3 * k + 2];
                if (blend) {
                    const float bonus = blend[2 * n], flash = blend[2 * n + 1];
                    r = blended_channel((unsigned char)r, 0, bonus, flash); g = blended_channel((unsigned char)g, 1, bonus, flash); b = blended_channel((unsigned char)b, 2, bonus, flash);
                }
                pal[k] = (r | (g << 8) | (b << 16)) ^ 0x808080u;
            }
            __syncthreads();
            if constexpr (!FEW) {
                for (int k = threadIdx.x; k < 256 * COPIES / 4; k += OBS_THREADS) {
                    const unsigned int colour = pal[k / (COPIES / 4)];
                    reinterpret_cast<uint4 *>(copies)[k] = make_uint4(colour, colour, colour, colour);
                }
                __syncthreads();
            }
        }
        const bool resets = reset_mask && reset_mask[n];
        int low[TILES][3], high[TILES][3];      // the sums along the rows, a byte each of four rows a word
        const int4v start = {20 * 80 * 128 + 800, 20 * 80 * 128 + 800, 20 * 80 * 128 + 800, 20 * 80 * 128 + 800};      // the colours' 128, and half of 1600
        auto down_columns = [&](int half) __attribute__((always_inline)) {
            int4v total[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int4v upper = __builtin_amdgcn_mfma_i32_16x16x64_i8(down[half], int4v{high[2 * half][c], high[2 * half + 1][c], high[2 * half + 2][c], 0}, int4v{0, 0, 0, 0}, 0, 0, 0);
                total[c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(down[half], int4v{low[2 * half][c], low[2 * half + 1][c], low[2 * half + 2][c], 0}, start, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) total[c][r] = (upper[r] << 8) + total[c][r];
            }
            unsigned char *out = reinterpret_cast<unsigned char *>(gray_words[task & 1]) + (half * OBS_TILE + 4 * group) * GD_OBS_SIZE + wave * OBS_TILE + column;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // v / 1600 for v <= 1600 * 255 + 800: 2684355 is 2^32 / 1600 and 0.44 more, which takes v / 1600 up by less than 1 / 1600
                const unsigned int red = __umulhi((unsigned)total[0][r], 2684355u), green = __umulhi((unsigned)total[1][r], 2684355u), blue = __umulhi((unsigned)total[2][r], 2684355u);
                const unsigned int gray = __umul24(red, 77u << 8) + __umul24(green, 150u << 8) + __umul24(blue, 29u << 8) + (128u << 8);
                if (4 * group + r < OBS_TILE && column < OBS_TILE) out[r * GD_OBS_SIZE] = (unsigned char)(gray >> 16);
            }
        };
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            if constexpr (!FEW) pixels[(t + AHEAD) % TILES] = load_tile(task + (t + AHEAD) / TILES, (t + AHEAD) % TILES);
            const unsigned int word[4] = {pixels[t].x, pixels[t].y, pixels[t].z, pixels[t].w};
            int4v channel[3];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const unsigned int c0 = colour_of(word[j], 0), c1 = colour_of(word[j], 1), c2 = colour_of(word[j], 2), c3 = colour_of(word[j], 3);
                const unsigned int front = __builtin_amdgcn_perm(c1, c0, 0x05010400u), back = __builtin_amdgcn_perm(c3, c2, 0x05010400u);   // two reds, two greens
                channel[0][j] = (int)__builtin_amdgcn_perm(back, front, 0x05040100u);
                channel[1][j] = (int)__builtin_amdgcn_perm(back, front, 0x07060302u);
                channel[2][j] = (int)__builtin_amdgcn_perm(__builtin_amdgcn_perm(c3, c2, 0x06020602u), __builtin_amdgcn_perm(c1, c0, 0x06020602u), 0x05040100u);
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int4v sums = __builtin_amdgcn_mfma_i32_16x16x64_i8(channel[c], along, int4v{128, 128, 128, 128}, 0, 0, 0);   // 128 more: the byte above rounds
                const unsigned int front = __builtin_amdgcn_perm((unsigned)sums[1], (unsigned)sums[0], 0x05010400u), back = __builtin_amdgcn_perm((unsigned)sums[3], (unsigned)sums[2], 0x05010400u);
                low[t][c] = (int)(__builtin_amdgcn_perm(back, front, 0x05040100u) ^ 0x80808080u);
                high[t][c] = (int)__builtin_amdgcn_perm(back, front, 0x07060302u);
                if ((FEW || 16 * t >= VH % OBS_SOURCE_ROWS) && tile_row(block, t) >= source_rows) { low[t][c] = 0; high[t][c] = (int)0xD8D8D8D8u; }   // black: 80 * -128 = 256 * -40
            }
            if (t == 2) down_columns(0);
            if (t == 4) down_columns(1);      // not reached by three tiles
        }
        // the stack words that the roll keeps
        constexpr int WORDS = ROWS * GD_OBS_SIZE / 4, ROUNDS = (WORDS + OBS_THREADS - 1) / OBS_THREADS;
        const size_t first_word = (size_t)block * WORDS;
        unsigned int kept[ROUNDS][GD_FRAME_STACK];
#pragma unroll
        for (int j = 0; j < ROUNDS; ++j) {
            const int k = threadIdx.x + j * OBS_THREADS;
#pragma unroll
            for (int f = 0; f < GD_FRAME_STACK; ++f) {
                if constexpr (FEW) kept[j][f] = early[f];
                else kept[j][f] = k < WORDS && frames && !resets ? load_word(frames + ((size_t)n * GD_FRAME_STACK * F + f * F + first_word + k) * 4, stack_aligned) : 0u;
            }
        }
        __syncthreads();
        // the block's pixels are contiguous in the observation; they go out, and the stack is rolled, a word (four pixels) per thread
#pragma unroll
        for (int j = 0; j < ROUNDS; ++j) {
            const int k = threadIdx.x + j * OBS_THREADS;
            if (k >= WORDS) break;
            const unsigned int grays = gray_words[task & 1][k];
            const size_t word = first_word + k;
            if (obs) {
                unsigned char *out = obs + ((size_t)n * F + word) * 4;
                if ((reinterpret_cast<size_t>(obs) & 3) == 0) *reinterpret_cast<unsigned int *>(out) = grays;
                else for (int b = 0; b < 4; ++b) out[b] = (unsigned char)(grays >> (8 * b));
            }
            // a stack is [4][84][84] bytes, so word access only needs the tensors themselves word aligned
            if (frames) store_stack_word(frames + (size_t)n * GD_FRAME_STACK * F * 4, final_frames ? final_frames + (size_t)n * GD_FRAME_STACK * F * 4 : nullptr,
                                         final_hwc, stack_aligned, word, kept[j], grays, resets, stack_mode);
        }
    }
}

// `count` frames that lie `stride` bytes apart pooled to observations and stacks.
void launch_observe(hipStream_t stream, const unsigned char *indexed, size_t stride, int source_rows, const unsigned char *playpal, int count, unsigned char *obs, unsigned char *frames,
                    const unsigned char *reset_mask, int stack_mode, unsigned char *final_frames, bool final_hwc, const float *blend) {
    const bool few = observe_few(count), aligned = (reinterpret_cast<size_t>(indexed) & 15) == 0;
    auto kernel = few ? (aligned ? observe_kernel<true, true> : observe_kernel<false, true>) : (aligned ? observe_kernel<true, false> : observe_kernel<false, false>);
    const int groups = few ? count * (GD_OBS_SIZE / OBS_TILE) : observe_groups(count * OBS_BLOCKS);
    hipLaunchKernelGGL(kernel, dim3(groups), dim3(OBS_THREADS), 0, stream, indexed, stride, source_rows, playpal, count, obs, frames, reset_mask, stack_mode, final_frames, final_hwc, blend);
}

// engine.py:15381-15384: PLAYPAL expansion.  A thread takes sixteen pixels: one 16-byte load, sixteen palette words from LDS; the 48 bytes
// they make go through LDS, so that every store of a wavefront is a kilobyte of one piece (which host memory over PCIe asks for
// even more than device memory does: viewers have their frames expanded straight into pinned host memory).  512 lanes: bytes stored
// three apart took 0.123 ms, four times what the copy of as many bytes takes.
#define EXPAND_THREADS 192       // 3072 pixels: 25 blocks are exactly a lane's frame, so a block has one palette
#define EXPAND_PIXELS (EXPAND_THREADS * 16)
static_assert((GD_SCREEN_HEIGHT * SW) % EXPAND_PIXELS == 0, "expand_rgb_kernel: one lane per block");
__global__ void __launch_bounds__(EXPAND_THREADS) expand_rgb_kernel(const unsigned char *indexed, const unsigned char *playpal, size_t pixels, unsigned char *rgb,
                                                                    const float *blend, size_t lane_pixels) {
    __shared__ unsigned int pal[256];
    __shared__ __align__(16) unsigned int staged[EXPAND_THREADS / 64][64 * 12];
    const size_t block_first = (size_t)blockIdx.x * EXPAND_PIXELS;
    const int lane = blend ? (int)(block_first / lane_pixels) : 0;
    for (int k = threadIdx.x; k < 256; k += EXPAND_THREADS) {
        unsigned int r = playpal[3 * k], g = playpal[3 * k + 1], b = playpal[3 * k + 2];
        if (blend) {
            const float bonus = blend[2 * lane], flash = blend[2 * lane + 1];
            r = blended_channel((unsigned char)r, 0, bonus, flash); g = blended_channel((unsigned char)g, 1, bonus, flash); b = blended_channel((unsigned char)b, 2, bonus, flash);
        }
        pal[k] = r | (g << 8) | (b << 16);
    }
    __syncthreads();
    const size_t first = block_first + (size_t)threadIdx.x * 16;     // pixel counts are whole rows: a thread has all its sixteen or none
    const int wave = threadIdx.x >> 6, lane_id = threadIdx.x & 63;
    const bool aligned = ((reinterpret_cast<size_t>(indexed) | reinterpret_cast<size_t>(rgb)) & 15) == 0;
    if (!aligned) {
        if (first < pixels) for (int k = 0; k < 16; ++k) {
            const unsigned int c = pal[indexed[first + k]];
            rgb[(first + k) * 3] = (unsigned char)c; rgb[(first + k) * 3 + 1] = (unsigned char)(c >> 8); rgb[(first + k) * 3 + 2] = (unsigned char)(c >> 16);
        }
        return;
    }
    uint4 four = make_uint4(0u, 0u, 0u, 0u);
    if (first < pixels) four = *reinterpret_cast<const uint4 *>(indexed + first);
    const unsigned int words[4] = {four.x, four.y, four.z, four.w};
    unsigned int *mine = staged[wave] + lane_id * 12;
#pragma unroll
    for (int j = 0; j < 4; ++j) {   // four pixels, twelve bytes, three words
        const unsigned int c0 = pal[words[j] & 255u], c1 = pal[(words[j] >> 8) & 255u], c2 = pal[(words[j] >> 16) & 255u], c3 = pal[words[j] >> 24];
        mine[3 * j] = c0 | (c1 << 24); mine[3 * j + 1] = (c1 >> 8) | (c2 << 16); mine[3 * j + 2] = (c2 >> 16) | (c3 << 8);
    }
    wave_lds_fence();
    const size_t wave_bytes = (block_first + (size_t)wave * 1024) * 3, end = pixels * 3;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int at = j * 64 + lane_id;
        if (wave_bytes + (size_t)at * 16 < end) *reinterpret_cast<uint4 *>(rgb + wave_bytes + (size_t)at * 16) = reinterpret_cast<const uint4 *>(staged[wave])[at];
    }
}

// ---------------------------------------------------------------------------------------------
// finish: everything after the wall traversal and the flat selection, for one band of one lane's frame at a time,
// with the band held in LDS from the first shaded pixel to the pooled observation: plane and tier pixels
// (engine.py:13372-13405), the flat pass's pixels where nothing else shows (engine.py:11145-11163), billboards
// (engine.py:14762-14947), weapon and status bar (engine.py:15051-15110, 15232-15267), PLAYPAL expansion
// (engine.py:15381-15398), area pooling and the frame stack (_triton_kernels.py:120-177, engine.py:9545-9548).
// The 320x240 frame only goes to device memory when the caller asks for it.
// ---------------------------------------------------------------------------------------------
// A band is 80 frame rows: 28 observation rows pool exactly those (84 observation rows x 240 / 84 source rows each).
#define BAND_ROWS 80
#define BAND_COUNT (GD_SCREEN_HEIGHT / BAND_ROWS)
#define BAND_OBS_ROWS (BAND_ROWS * GD_OBS_SIZE / GD_SCREEN_HEIGHT)
#define BAND_THREADS 512   // sixteen wavefronts a compute unit when two work-groups share it: four per SIMD, none left over
static_assert(BAND_COUNT * BAND_ROWS == GD_SCREEN_HEIGHT && BAND_OBS_ROWS * BAND_COUNT == GD_OBS_SIZE, "bands tile the frame and the observation");
static_assert(BAND_THREADS >= SW && (BAND_OBS_ROWS * GD_OBS_SIZE) % 4 == 0, "band_finish_kernel: thread layout");

struct BandFrame {   // the rows [row0, row0 + BAND_ROWS) of a lane's frame, in LDS
    unsigned char *rows;
    int row0;
    __device__ __forceinline__ unsigned char *at(int y, int x) const { return rows + (y - row0) * SW + x; }
};

struct FinishOut {   // device pointers of the chunk's first lane; null = not wanted
    unsigned char *indexed, *rgb, *obs, *frames, *final_frames;
    const unsigned char *reset_mask;
    const float *blend;
    int stack_mode, source_rows;
    bool final_hwc;
};

__global__ void __launch_bounds__(BAND_THREADS) __attribute__((amdgpu_waves_per_eu(4, 4))) band_finish_kernel(DeviceMap dm, Overlays ov, gd_lanes_desc lanes, int lane_base, int lane_count, Scratch sc, FinishOut out) {
    extern __shared__ unsigned char shared_raw[];                // billboard records, when there are too many to reuse the tables' LDS
    __shared__ unsigned int band_words[BAND_ROWS * SW / 4];
    // the sector table and the colormap serve the shading phase only; the billboard records take their place afterwards
    __shared__ struct { float4 sector[LDS_SECTORS]; unsigned char colormap[32 * 256]; } shading_lds;
    float4 *sector_lds = shading_lds.sector;
    unsigned char *colormap_lds = shading_lds.colormap;
    __shared__ unsigned int sector_level_lds[LDS_SECTORS];
    __shared__ TexLds tex_lds;
    __shared__ i64 level_plane_lds[2 * PLANE_LEVELS * 2];
    __shared__ i64 step_scale_lds[STEP_TABLE];
    __shared__ unsigned int pal[256];                            // PLAYPAL after the lane's screen blend: red | green << 8 | blue << 16
    __shared__ unsigned int gray_words[BAND_OBS_ROWS * GD_OBS_SIZE / 4];
    __shared__ int on_screen_count;
    const gd_map_desc *m = &dm.d;
    const int band = blockIdx.x, local = blockIdx.y;
    if (local >= lane_count) return;     // uniform over the block
    const int n = lane_base + local;
    const int tid = threadIdx.x;
    const int row0 = band * BAND_ROWS;
    const int view_rows = row0 >= VH ? 0 : (row0 + BAND_ROWS <= VH ? BAND_ROWS : VH - row0);   // the rest are status bar rows
    unsigned char *band_bytes = reinterpret_cast<unsigned char *>(band_words);
    BandFrame frame; frame.rows = band_bytes; frame.row0 = row0;
    Tables tb;
    stage_tables(m, sector_lds, &tex_lds, tb);
    for (int k = tid; k < 32 * 256 / 4; k += BAND_THREADS) reinterpret_cast<unsigned int *>(colormap_lds)[k] = reinterpret_cast<const unsigned int *>(m->colormap)[k];
    const int floors = m->floor_level_count, levels = floors + m->ceil_level_count;
    const bool tabled = dm.sector_level != nullptr;
    const bool levels_staged = levels <= 2 * PLANE_LEVELS;
    if (tabled) {
        for (int s = tid; s < tb.sector_cached; s += BAND_THREADS) sector_level_lds[s] = dm.sector_level[s];
        if (levels_staged) for (int k = tid; k < 2 * levels; k += BAND_THREADS) level_plane_lds[k] = sc.level_plane[(size_t)local * levels * 2 + k];
        if (tid < STEP_TABLE) step_scale_lds[tid] = sc.step_scale[(size_t)local * STEP_TABLE + tid];
    }
    if (tid < 256) {
        unsigned int r = m->playpal[3 * tid], g = m->playpal[3 * tid + 1], b = m->playpal[3 * tid + 2];
        if (out.blend) {
            const float bonus = out.blend[2 * local], flash = out.blend[2 * local + 1];
            r = blended_channel((unsigned char)r, 0, bonus, flash); g = blended_channel((unsigned char)g, 1, bonus, flash); b = blended_channel((unsigned char)b, 2, bonus, flash);
        }
        pal[tid] = r | (g << 8) | (b << 16);
    }
    if (tid == 0) on_screen_count = 0;
    __syncthreads();
    const LaneCtx L = sc.ctx[local];
    LaneTables lt; lt.step_scale = step_scale_lds; lt.floors = floors;
    lt.level_plane = levels_staged ? level_plane_lds : sc.level_plane + (size_t)local * levels * 2;
    // --- the status bar rows of this band (engine.py:15232-15267); empty without status bar patches
    if (view_rows < BAND_ROWS && lanes.hud_state && ov.d.hud_patch_count > 0) {
        static_assert(BAND_ROWS - VH % BAND_ROWS == HUD_ROWS, "the last band holds the status bar");
        for (int tile = tid >> 6; tile < HUD_TILES; tile += BAND_THREADS / 64)
            hud_tile(ov.d, lanes.hud_state + (size_t)n * 9, tile, [&](int x, int y, unsigned char value) { band_bytes[(view_rows + y) * SW + x] = value; });
    } else {
        for (int p = tid; p < (BAND_ROWS - view_rows) * SW; p += BAND_THREADS) band_bytes[view_rows * SW + p] = 0;
    }
    // --- every view pixel of the band once: a wall tier's palette index, a visplane's flat, a masked mid-texture's texel, or
    // the flat pass's pick.  A wavefront takes a row at a time, its lanes the row's five groups of 64 columns: what depends
    // on the row alone is worked out once per row, and each stage's loads are issued together.
    const size_t lane_pixels = (size_t)local * VH * SW;
    const int wave = tid >> 6, lane_id = tid & 63;
    constexpr int ROW_GROUPS = SW / 64;
    for (int py = wave; py < view_rows; py += BAND_THREADS / 64) {
        const int y = row0 + py;
        const size_t row_at = lane_pixels + (size_t)y * SW;
        const i64 yslope = sc.row_slope[(size_t)local * VH + y];
        unsigned int meta[ROW_GROUPS];
#pragma unroll
        for (int j = 0; j < ROW_GROUPS; ++j) meta[j] = sc.meta[row_at + j * 64 + lane_id];
        int colormap_row[ROW_GROUPS]; unsigned char texel[ROW_GROUPS];
        bool shade[ROW_GROUPS];
#pragma unroll
        for (int j = 0; j < ROW_GROUPS; ++j) {
            const int ps = (int)((meta[j] >> META_SECTOR_SHIFT) & META_SECTOR_MASK) - 1;
            shade[j] = tabled && ps >= 0 && !(meta[j] & (META_FILLED | META_MASKED));
            texel[j] = 0; colormap_row[j] = 0;
            if (!shade[j]) continue;
            const bool is_floor = (meta[j] & META_FLOOR) != 0;
            const unsigned int pair = ps < tb.sector_cached ? sector_level_lds[ps] : dm.sector_level[ps];
            const size_t texel_at = flat_sample_tabled(tb, L, lt, yslope, is_floor ? (pair & 0xFFFF) : (pair >> 16), ps, is_floor, j * 64 + lane_id, y, &colormap_row[j]);
            texel[j] = m->tex_atlas[texel_at];
        }
#pragma unroll
        for (int j = 0; j < ROW_GROUPS; ++j) {
            const int x = j * 64 + lane_id;
            const int ps = (int)((meta[j] >> META_SECTOR_SHIFT) & META_SECTOR_MASK) - 1;
            unsigned char colour;
            if (meta[j] & META_MASKED) colour = sc.masked_texel[row_at + x];   // left there by masked_midtexture
            else if (meta[j] & META_FILLED) colour = (unsigned char)(meta[j] >> META_SECTOR_SHIFT);
            else if (shade[j]) colour = colormap_lds[colormap_row[j] * 256 + texel[j]];
            else if (ps >= 0) colour = flat_pixel(tb, colormap_lds, L, ps, (meta[j] & META_FLOOR) != 0, x, y);
            else colour = flat_pixel(tb, colormap_lds, L, sc.flat_sector[row_at + x], ((float)y - flat_center(L)) > 0, x, y);   // the flat pass's picture
            band_bytes[py * SW + x] = colour;
        }
    }
    // --- billboards, one thread per screen column
    if (lanes.sprite_slots > 0 && lanes.sprite_x && view_rows > 0) {
        __syncthreads();                  // every shaded pixel is in place, and the shading tables are free
        const bool fits = (size_t)lanes.sprite_slots * sizeof(SpriteRec) <= sizeof(shading_lds);
        SpriteRec *sp = reinterpret_cast<SpriteRec *>(fits ? reinterpret_cast<unsigned char *>(&shading_lds) : shared_raw);
        stage_sprites(dm, lanes, n, L, 0, SW, row0, row0 + view_rows, sp, &on_screen_count);
        __syncthreads();
        if (tid < SW && on_screen_count > 0) sprite_column(dm, lanes, sc, local, n, L, sp, on_screen_count, tid, row0, row0 + view_rows, frame);
    }
    __syncthreads();
    // --- the player's weapon and its muzzle flash (engine.py:15051-15110)
    if (lanes.weapon_state && ov.d.weapon_patch_count > 0) {
        const int64_t *state = lanes.weapon_state + (size_t)n * 5;
        if (state[4] != 0) {
            const Psprite weapon(ov.d, state[0], state[2], state[3]), flash(ov.d, state[1], state[2], state[3]);
            int x0 = SW, y0 = VH, x1 = 0, y1 = 0;
            weapon.bounds(x0, y0, x1, y1); flash.bounds(x0, y0, x1, y1);
            for (int py = max(y0, row0) + wave; py < min(y1, row0 + view_rows); py += BAND_THREADS / 64) {
                for (int px = x0 + lane_id; px < x1; px += 64) Psprite::paint(ov.d, weapon, flash, px, py, band_bytes + (py - row0) * SW + px);
            }
        }
        __syncthreads();
    }
    // --- what the caller asked for
    if (out.indexed) {
        uint4 *rows = reinterpret_cast<uint4 *>(out.indexed + ((size_t)local * GD_SCREEN_HEIGHT + row0) * SW);
        const bool aligned = (reinterpret_cast<size_t>(out.indexed) & 15) == 0;
        if (aligned) {
            for (int k = tid; k < BAND_ROWS * SW / 16; k += BAND_THREADS) rows[k] = reinterpret_cast<const uint4 *>(band_words)[k];
        } else {
            unsigned char *bytes = out.indexed + ((size_t)local * GD_SCREEN_HEIGHT + row0) * SW;
            for (int k = tid; k < BAND_ROWS * SW; k += BAND_THREADS) bytes[k] = band_bytes[k];
        }
    }
    if (out.rgb) {   // four pixels, twelve bytes, three words per step
        unsigned char *rows = out.rgb + ((size_t)local * GD_SCREEN_HEIGHT + row0) * SW * 3;
        const bool aligned = (reinterpret_cast<size_t>(out.rgb) & 3) == 0;
        for (int k = tid; k < BAND_ROWS * SW / 4; k += BAND_THREADS) {
            const unsigned int four = band_words[k];
            const unsigned int c0 = pal[four & 0xFFu], c1 = pal[(four >> 8) & 0xFFu], c2 = pal[(four >> 16) & 0xFFu], c3 = pal[four >> 24];
            const unsigned int w0 = c0 | (c1 << 24), w1 = (c1 >> 8) | (c2 << 16), w2 = (c2 >> 16) | (c3 << 8);
            if (aligned) {
                unsigned int *words = reinterpret_cast<unsigned int *>(rows) + 3 * k;
                words[0] = w0; words[1] = w1; words[2] = w2;
            } else {
                unsigned char *bytes = rows + 12 * k;
                for (int q = 0; q < 4; ++q) { bytes[q] = (unsigned char)(w0 >> (8 * q)); bytes[4 + q] = (unsigned char)(w1 >> (8 * q)); bytes[8 + q] = (unsigned char)(w2 >> (8 * q)); }
            }
        }
    }
    if (!out.obs && !out.frames) return;
    // --- the band's observation rows, pooled from LDS (_triton_kernels.py:120-177).  An observation pixel covers 240/84 source
    // rows and 320/84 source columns; its weights (y_overlap * x_overlap) // 48 are exactly (y_overlap / 12) * (x_overlap / 4),
    // since row overlaps are multiples of 12 and column overlaps multiples of 4 (84 = 12 * 7 = 4 * 21, 240 = 12 * 20,
    // 320 = 4 * 80): the weighted sum factors into a pass along the rows and one down the columns, all in integers.
    // Seven observation rows pool exactly twenty source rows; rows at or past source_rows are black.
    constexpr int OBS_GROUP = 7, SRC_GROUP = OBS_GROUP * GD_SCREEN_HEIGHT / GD_OBS_SIZE;   // 7 and 20
    static_assert(BAND_OBS_ROWS % OBS_GROUP == 0 && SRC_GROUP * GD_OBS_SIZE == OBS_GROUP * GD_SCREEN_HEIGHT, "observation rows group by seven");
    // per source row and observation column: the three channel sums along the row, 16 bits each (at most 80 * 255)
    unsigned short *along = reinterpret_cast<unsigned short *>(&shading_lds);
    static_assert(sizeof(shading_lds) >= (size_t)SRC_GROUP * GD_OBS_SIZE * 3 * sizeof(unsigned short), "row sums fit the shading tables' LDS");
    const int first_obs_row = band * BAND_OBS_ROWS;
    for (int group = 0; group < BAND_OBS_ROWS / OBS_GROUP; ++group) {
        __syncthreads();   // the billboard records (first round) or the last group's row sums are no longer needed
        for (int q = tid; q < SRC_GROUP * GD_OBS_SIZE; q += BAND_THREADS) {
            const int sy = q / GD_OBS_SIZE, ox = q - sy * GD_OBS_SIZE;
            const int band_row = group * SRC_GROUP + sy;
            const unsigned char *row = band_bytes + band_row * SW;
            const int x_start = ox * 320, x_end = x_start + 320, first_x = x_start / 84;
            unsigned int rs = 0, gs = 0, bs = 0;
            if (row0 + band_row < out.source_rows) {
#pragma unroll
                for (int sx = 0; sx < 5; ++sx) {
                    const int source_x = first_x + sx;
                    const int over = min(x_end, (source_x + 1) * 84) - max(x_start, source_x * 84);
                    const unsigned weight = (source_x >= SW || over <= 0) ? 0u : (unsigned)over >> 2;
                    const unsigned int colour = pal[row[min(source_x, SW - 1)]];
                    rs += __umul24(colour & 0xFFu, weight); gs += __umul24((colour >> 8) & 0xFFu, weight); bs += __umul24(colour >> 16, weight);
                }
            }
            along[3 * q] = (unsigned short)rs; along[3 * q + 1] = (unsigned short)gs; along[3 * q + 2] = (unsigned short)bs;
        }
        __syncthreads();
        for (int q = tid; q < OBS_GROUP * GD_OBS_SIZE; q += BAND_THREADS) {
            const int row_in_group = q / GD_OBS_SIZE, ox = q - row_in_group * GD_OBS_SIZE;
            const int y_start = row_in_group * 240, y_end = y_start + 240, first_y = y_start / 84;   // relative to the group's first source row
            unsigned int rs = 0, gs = 0, bs = 0;
#pragma unroll
            for (int sy = 0; sy < 4; ++sy) {
                const int source_y = first_y + sy;
                const int over = min(y_end, (source_y + 1) * 84) - max(y_start, source_y * 84);
                const unsigned weight = (source_y >= SRC_GROUP || over <= 0) ? 0u : (unsigned)over / 12u;
                const unsigned short *sums = along + 3 * (min(source_y, SRC_GROUP - 1) * GD_OBS_SIZE + ox);
                rs += __umul24(sums[0], weight); gs += __umul24(sums[1], weight); bs += __umul24(sums[2], weight);
            }
            const unsigned r = (rs + 800u) / 1600u, g = (gs + 800u) / 1600u, b = (bs + 800u) / 1600u;
            reinterpret_cast<unsigned char *>(gray_words)[group * OBS_GROUP * GD_OBS_SIZE + q] = (unsigned char)((r * 77u + g * 150u + b * 29u + 128u) >> 8);
        }
    }
    __syncthreads();
    // the band's pixels are contiguous in the observation; they go out, and the stack is rolled, a word (four pixels) per thread
    const size_t F = (size_t)GD_OBS_SIZE * GD_OBS_SIZE / 4;     // words per observation
    const bool stack_aligned = ((reinterpret_cast<size_t>(out.frames) | reinterpret_cast<size_t>(out.final_frames)) & 3) == 0;
    const bool resets = out.reset_mask && out.reset_mask[local];
    auto load_word = [](const unsigned char *p, bool aligned) -> unsigned int {
        if (aligned) return *reinterpret_cast<const unsigned int *>(p);
        return (unsigned)p[0] | ((unsigned)p[1] << 8) | ((unsigned)p[2] << 16) | ((unsigned)p[3] << 24);
    };
    auto store_word = [](unsigned char *p, unsigned int v, bool aligned) {
        if (aligned) *reinterpret_cast<unsigned int *>(p) = v;
        else for (int k = 0; k < 4; ++k) p[k] = (unsigned char)(v >> (8 * k));
    };
    for (int k = tid; k < BAND_OBS_ROWS * GD_OBS_SIZE / 4; k += BAND_THREADS) {
        const size_t word = (size_t)first_obs_row * GD_OBS_SIZE / 4 + k;
        const unsigned int grays = gray_words[k];
        if (out.obs) store_word(out.obs + ((size_t)local * F + word) * 4, grays, (reinterpret_cast<size_t>(out.obs) & 3) == 0);
        if (!out.frames) continue;
        unsigned char *stack_lane = out.frames + (size_t)local * GD_FRAME_STACK * F * 4;
        unsigned int kept[GD_FRAME_STACK];
        // a lane that steps drops its oldest observation; it is only read for a copy of a stack that stays as it is
        const bool reads = !resets, reads_oldest = reads && out.stack_mode != GD_STACK_STEP && out.final_frames;
        for (int f = 0; f < GD_FRAME_STACK; ++f)
            kept[f] = (reads && (f > 0 || reads_oldest)) ? load_word(stack_lane + (size_t)f * F * 4 + word * 4, stack_aligned) : 0u;
        store_stack_word(stack_lane, out.final_frames ? out.final_frames + (size_t)local * GD_FRAME_STACK * F * 4 : nullptr, out.final_hwc,
                         stack_aligned, word, kept, grays, resets, out.stack_mode);
    }
}

// ---------------------------------------------------------------------------------------------
// actor packing: engine.py:14328-14682 with the sprite-id helpers of 14011-14136 and 14258-14317
// ---------------------------------------------------------------------------------------------
// Index of the animation frame showing after `elapsed` tics: the number of frames whose running end has
// passed, held on the last one (engine.py:14084-14091, 14117-14122).
__device__ __forceinline__ int frame_after(i64 elapsed, const int64_t *durations, int frames, i64 count) {
    i64 end = 0; int frame = 0;
    for (int k = 0; k < frames; ++k) { end += durations[k]; frame += elapsed >= end ? 1 : 0; }
    const i64 last = count - 1;
    return (int)(frame < last ? frame : last);
}

__device__ __forceinline__ i64 clamp_type(i64 v, i64 hi) { return v < 0 ? 0 : (v > hi ? hi : v); }

__device__ __forceinline__ i64 explosion_patch(const gd_actor_desc &a, i64 kind, i64 remaining) {
    kind = clamp_type(kind, 2);
    const int F = a.explosion_frames;
    const i64 elapsed = a.projectile_explosion_total_tics[kind] - remaining;
    const int frame = frame_after(elapsed, a.projectile_explosion_frame_durations + kind * F, F, a.projectile_explosion_frame_counts[kind]);
    return a.raw_projectile_explosion_sprite_ids[kind * F + frame];
}

// Doom's clockwise 1..8 sprite rotation as 0..7 (engine.py:13994-14009) of an actor at (x, y) that faces `heading`, one rounded operation at a
// time as Torch evaluates the expression on a device, where a tensor over a number is multiplied by the number's reciprocal.
__device__ __forceinline__ int facing_of(const gd_facing_desc &f, int n, float x, float y, float heading) {
    const float TWO_PI = (float)(2.0 * 3.14159265358979323846), EIGHTH_PI = (float)(3.14159265358979323846 / 8), PER_QUARTER_PI = 1.0f / (float)(3.14159265358979323846 / 4);
    float turn = fmodf((atan2f(f.y[n] - y, f.x[n] - x) - heading) + EIGHTH_PI, TWO_PI);
    if (turn != 0.0f && turn < 0.0f) turn += TWO_PI;         // torch.remainder with a positive divisor
    return (int)((i64)floorf(turn * PER_QUARTER_PI) & 7);
}

// FACING: rotations are worked out here (gd_pack_actors_facing), not read.  As Torch operators they were some forty kernels, and the copies of
// the map's columns and the weapon's words a dozen more: with them an engine's frame of 2048 lanes took 2484 us, of one lane (which the host's
// launches take longest for) 619 us; without 2229 and 303 us.  This kernel takes 29 us at 2048 lanes of 495 slots, 26 where it reads rotations.
template <bool FACING>
__global__ void __launch_bounds__(64) pack_actors_kernel(gd_actor_desc a, gd_facing_desc f, int width) {
    const int slot = blockIdx.x * blockDim.x + threadIdx.x;
    const int n = blockIdx.y;
    if (slot >= width || n >= a.lane_count) return;
    float x = 0, y = 0, z = 0; i64 patch = 0; bool alive = false, bright = false; int style = -1;
    int k = slot;
    const int Se = a.enemy_slots, Sd = a.doll_count, Sp = a.player_projectile_slots, Sq = a.enemy_projectile_slots;
    if (k < Se) {                                   // monsters (engine.py:14011-14077, 14125-14136)
        const size_t i = (size_t)n * Se + k;
        x = a.enemy_x[i]; y = a.enemy_y[i]; z = a.enemy_z[i]; alive = a.enemy_alive[i] != 0;
        const i64 kind = clamp_type(a.enemy_type[i], 5);
        const int facing = FACING ? facing_of(f, n, x, y, f.enemy_angle[i]) : a.enemy_rotation[i];
        const int tics = a.enemy_animation_tics[i];
        int walking = (tics / a.enemy_walk_frame_tics[kind]) % 4;
        int idling = (tics / a.enemy_idle_frame_tics[kind]) % 2;
        if (kind == 2) idling = 0;
        if (a.enemy_target_slot[i] < -1) walking = idling;
        const int phase = a.enemy_attack_phase[i], cooldown = a.enemy_cooldown[i];
        const bool recovering = cooldown > a.enemy_attack_recovery[kind] / 2;
        const bool hitscanner = kind == 0 || kind == 1, melee = kind == 4 || kind == 5;
        int attacking = 0;
        if (hitscanner && phase == 2) attacking = recovering ? 1 : 0;
        if (melee && phase == 1) attacking = cooldown <= 8 ? 1 : 0;
        if (melee && phase == 2) attacking = 2;
        if (kind == 3 && (phase == 4 || phase == 2)) attacking = 1;
        if (kind == 3 && phase == 3) attacking = 2;
        patch = phase > 0 ? a.enemy_attack_sprite_ids[(kind * a.attack_frames + attacking) * 8 + facing]
                          : a.enemy_walk_sprite_ids[(kind * 4 + walking) * 8 + facing];
        if (a.enemy_pain_tics[i] > 0) patch = a.enemy_pain_sprite_ids[kind * 8 + facing];
        bright = (kind == 1 && phase == 2 && recovering) || (kind == 3 && (phase == 2 || phase == 3));
    } else if ((k -= Se) < Sd) {                    // the other players' start dolls (engine.py:14345-14379)
        const size_t row = FACING ? (size_t)k * f.doll_stride : k;
        x = a.doll_x[row]; y = a.doll_y[row]; z = a.doll_z[k]; alive = a.player_dead[n] == 0;
        const int facing = FACING ? facing_of(f, n, x, y, f.doll_degrees[row] * (float)(3.14159265358979323846 / 180)) : a.doll_rotation[(size_t)n * Sd + k];
        patch = a.enemy_walk_sprite_ids[(2 * 4 + 0) * 8 + facing];
    } else if ((k -= Sd) < Se) {                    // corpses (engine.py:14079-14106)
        const size_t i = (size_t)n * Se + k;
        x = a.enemy_x[i]; y = a.enemy_y[i]; z = a.enemy_z[i]; alive = a.enemy_death_tics[i] > 0;
        const i64 kind = clamp_type(a.enemy_death_type[i], 5);
        const i64 elapsed = a.enemy_death_elapsed[i];
        if (a.enemy_death_extreme[i]) {
            const int F = a.xdeath_frames;
            patch = a.enemy_xdeath_sprite_ids[kind * F + frame_after(elapsed, a.enemy_xdeath_frame_durations + kind * F, F, a.enemy_xdeath_frame_counts[kind])];
        } else {
            const int F = a.death_frames;
            patch = a.enemy_death_sprite_ids[kind * F + frame_after(elapsed, a.enemy_death_frame_durations + kind * F, F, a.enemy_death_frame_counts[kind])];
        }
    } else if ((k -= Se) < Sp) {                    // rockets and plasma balls in flight (engine.py:14410-14460)
        const size_t i = (size_t)n * Sp + k;
        x = a.projectile_x[i]; y = a.projectile_y[i]; z = a.projectile_z[i]; alive = a.projectile_alive[i] != 0;
        const i64 shot = clamp_type(a.projectile_type[i], 1);
        const int frame = shot == 1 ? (a.projectile_age[i] / 6) % 2 : 0;
        const int facing = FACING ? facing_of(f, n, x, y, atan2f(f.projectile_velocity_y[i], f.projectile_velocity_x[i])) : a.projectile_rotation[i];
        patch = a.raw_projectile_flight_sprite_ids[(shot * 2 + frame) * 8 + facing];
        bright = alive; style = shot == 1 ? 0 : -1;
    } else if ((k -= Sp) < Sq) {                    // monster fireballs in flight (engine.py:14462-14510)
        const size_t i = (size_t)n * Sq + k;
        x = a.enemy_projectile_x[i]; y = a.enemy_projectile_y[i]; z = a.enemy_projectile_z[i]; alive = a.enemy_projectile_alive[i] != 0;
        const int frame = (a.enemy_projectile_age[i] / 4) % 2;
        const int facing = FACING ? facing_of(f, n, x, y, atan2f(f.enemy_projectile_velocity_y[i], f.enemy_projectile_velocity_x[i])) : a.enemy_projectile_rotation[i];
        patch = a.raw_projectile_flight_sprite_ids[(2 * 2 + frame) * 8 + facing];
        bright = alive; style = 1;
    } else if ((k -= Sq) < Sp) {                    // the player's explosions (engine.py:14512-14541)
        const size_t i = (size_t)n * Sp + k;
        x = a.projectile_x[i]; y = a.projectile_y[i]; z = a.projectile_z[i]; alive = a.projectile_impact_tics[i] > 0;
        patch = explosion_patch(a, a.projectile_impact_type[i], a.projectile_impact_tics[i]);
        bright = alive; style = a.projectile_impact_type[i] == 1 ? 0 : -1;
    } else if ((k -= Sp) < Sq) {                    // fireball explosions (engine.py:14543-14573)
        const size_t i = (size_t)n * Sq + k;
        x = a.enemy_projectile_x[i]; y = a.enemy_projectile_y[i]; z = a.enemy_projectile_z[i]; alive = a.enemy_projectile_impact_tics[i] > 0;
        patch = explosion_patch(a, 2, a.enemy_projectile_impact_tics[i]);
        bright = alive; style = 1;
    } else if ((k -= Sq) < a.fog_slots) {           // teleport fog: 12 frames of 6 tics out of 72 (engine.py:14577-14595)
        const size_t i = (size_t)n * a.fog_slots + k;
        x = a.teleport_fog_x[i]; y = a.teleport_fog_y[i]; z = a.teleport_fog_z[i];
        const int tics = a.teleport_fog_tics[i];
        alive = tics > 0;
        const int elapsed = 72 - tics;
        int frame = elapsed >= 0 ? elapsed / 6 : -((-elapsed + 5) / 6);   // floor division, like Torch's //
        if (frame > 11) frame = 11;
        if (frame < 0) frame += 12;                                      // a negative index counts from the end
        patch = a.raw_teleport_fog_sprite_ids[frame];
        bright = alive; style = 1;
    } else if ((k -= a.fog_slots) < a.puff_slots) { // bullet puffs: 4 frames of 4 tics (engine.py:14597-14630)
        const size_t i = (size_t)n * a.puff_slots + k;
        x = a.hitscan_puff_x[i]; y = a.hitscan_puff_y[i]; z = a.hitscan_puff_z[i];
        const int tics = a.hitscan_puff_tics[i];
        alive = tics > 0;
        const int frame = tics > 12 ? 0 : (tics > 8 ? 1 : (tics > 4 ? 2 : 3));
        patch = a.raw_bullet_puff_sprite_ids[frame];
        bright = frame == 0; style = -2;
    } else if ((k -= a.puff_slots) < a.item_count) {   // map items (engine.py:14258-14317, 14632-14655)
        const size_t i = (size_t)n * a.item_count + k;
        const size_t row = FACING ? (size_t)k * f.item_stride : k;
        x = a.item_x[row]; y = a.item_y[row]; z = a.item_z[k]; alive = a.item_available[i] != 0;
        const i64 kind = a.item_types[k];
        const i64 elapsed = (i64)a.episode_time[n] + (6 - (i64)a.item_animation_initial_tics[i]);
        const i64 sixth = elapsed >= 0 ? elapsed / 6 : -((-elapsed + 5) / 6);
        const int phase = (int)(((sixth % 6) + 6) % 6);
        const int swing = phase == 0 ? -1 : (phase <= 3 ? phase - 1 : 5 - phase);   // A, then B C D C B
        patch = a.item_raw_visual_types[k];
        if (kind == 2014 && swing >= 0) patch = a.raw_item_animation_sprite_ids[swing];
        if (kind == 2015 && swing >= 0) patch = a.raw_item_animation_sprite_ids[3 + swing];
        const bool green = kind == 2018 && (((elapsed % 13) + 13) % 13) >= 6;
        const bool blue = kind == 2019 && (((elapsed % 12) + 12) % 12) >= 6;
        if (green) patch = a.raw_item_animation_sprite_ids[6];
        if (blue) patch = a.raw_item_animation_sprite_ids[7];
        bright = green || blue;
    } else {                                        // what monsters drop (engine.py:14657-14682)
        k -= a.item_count;
        const size_t i = (size_t)n * a.drop_slots + k;
        x = a.drop_x[i]; y = a.drop_y[i]; z = a.drop_z[i];
        const i64 kind = a.drop_type[i];
        alive = kind >= 0 && a.drop_spawned[i] != 0;
        patch = a.raw_static_sprite_ids[kind == 2002 ? 14 : (kind == 2007 ? 6 : 12)];
    }
    const size_t out = (size_t)n * width + slot;
    a.sprite_x[out] = x; a.sprite_y[out] = y; a.sprite_z[out] = z;
    a.sprite_id[out] = (int)patch;
    a.sprite_alive[out] = alive ? 1 : 0; a.sprite_fullbright[out] = bright ? 1 : 0; a.sprite_style[out] = (signed char)style;
}

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
int fail(int code, const std::string &message) { return gd_fail(code, message); }

// gd_pack_weapon: one thread per lane.  Which patch the player's weapon shows and where (engine.py:14949-14967,
// 15051-15092): the frame table is indexed by weapon, by a parity that alternates with every shot (an idling chainsaw
// alternates every four tics instead) and by the tics left of the weapon's state; a weapon being lowered or raised sits
// six map pixels lower per tic, as does one raised at the start of an episode; a ready weapon sways with the player's bob
// along a circle of the fine sine table that advances 128 steps a tic.
__global__ void __launch_bounds__(64) pack_weapon_kernel(gd_weapon_desc d, unsigned narrow) {
    const int lane = blockIdx.x * blockDim.x + threadIdx.x;
    if (lane >= d.lane_count) return;
    // word k of the descriptor's nine, which is 32 bits wide where bit k of `narrow` is set
    const auto word = [&](const int64_t *words, int k) -> i64 { return (narrow >> k) & 1u ? reinterpret_cast<const int32_t *>(words)[lane] : words[lane]; };
    const i64 slots = d.cooldown_slots;
    const i64 weapon = clampi(word(d.active_weapon, 0), 0, 7);
    const i64 state_tics = word(d.weapon_state_cooldown, 1);
    const i64 tic = clampi(state_tics, 0, slots - 1);
    i64 parity = word(d.weapon_fire_count, 2) % 2;
    if (parity < 0) parity += 2;                    // torch.remainder: the sign of the divisor
    if (weapon == 1 && tic == 0) parity = (max64(word(d.weapon_ready_tics, 3) - 1, 0) / 4) % 2;
    const i64 entry = (weapon * 2 + parity) * slots + tic;
    const i64 switching = word(d.pending_weapon, 6) >= 0;
    const i64 raising = word(d.weapon_raise_cooldown, 5);
    i64 lowered = switching ? clampi(16 - word(d.weapon_lower_cooldown, 4), 0, 16) : raising;      // engine.py:111 (16 tics to lower)
    const i64 time = word(d.episode_time, 7);
    lowered = max64(lowered, clampi(14 - (time - 1), 0, 14));                                   // engine.py:114 (14 tics to raise at spawn)
    const bool steady = state_tics <= 0 && raising <= 0 && !switching;
    const i64 swing = mul64(time, 128) & (FINE_ANGLES - 1);
    const i64 bob = word(d.player_bob_fixed, 8);
    const i64 sway_x = steady ? mul64(bob, d.fine_sine[(swing + FINE_ANGLES / 4) & (FINE_ANGLES - 1)]) >> 16 : 0;
    const i64 sway_y = steady ? mul64(bob, d.fine_sine[swing & (FINE_ANGLES / 2 - 1)]) >> 16 : 0;
    int64_t *out = d.weapon_state + (size_t)lane * 5;
    out[0] = d.weapon_frame_ids[entry];
    out[1] = d.weapon_flash_ids[entry];
    out[2] = sway_x;
    out[3] = mul64(lowered, 6 * FIXED_UNIT) + sway_y;
    out[4] = d.player_dead[lane] ? 0 : 1;
    if (d.flash_light) d.flash_light[lane] = d.weapon_flash_lights[entry];
}

// gd_pack_decals: one wavefront per lane.  A slot's place is the number of slots before it in the order (a stable one), counted against
// 64 slots' keys in LDS at a time.  Each float operation is rounded on its own, as in the Torch expressions.  2048 lanes of 64 slots: some thirty
// Torch kernels, a sort among them, 0.20 ms; one kernel, 0.011 ms.
#define DECAL_FREE 2147483647LL      // the place in the order of a slot without an impact
__global__ void __launch_bounds__(64) pack_decals_kernel(const int64_t *serial, const int64_t *wall, const float *along, const float *impact_z, const int64_t *style,
                                                         const float *walls, int wall_count, const int64_t *fine_sine, int slots, int32_t *decal_state, float *decal_geom) {
    __shared__ i64 keys[64];
    const size_t lane = (size_t)blockIdx.x * (size_t)slots;
    const float TWO_PI = (float)(2.0 * 3.14159265358979323846), FINE_PER_RADIAN = (float)(FINE_ANGLES / (2.0 * 3.14159265358979323846));
    for (int base = 0; base < slots; base += 64) {
        const int s = base + (int)threadIdx.x;
        const bool held = s < slots;
        const i64 own = held ? serial[lane + s] : -1, key = own >= 0 ? own : DECAL_FREE;
        int place = 0;
        for (int other = 0; other < slots; other += 64) {
            const int j = other + (int)threadIdx.x;
            const i64 theirs = j < slots ? serial[lane + j] : -1;
            __syncthreads();
            keys[threadIdx.x] = theirs >= 0 ? theirs : DECAL_FREE;
            __syncthreads();
            const int count = min(64, slots - other);
            for (int k = 0; k < count; ++k) place += keys[k] < key || (keys[k] == key && other + k < s);
        }
        if (!held) continue;
        const i64 linedef = clampi(wall[lane + s], 0, wall_count - 1), kind = style[lane + s];
        const float4 ends = reinterpret_cast<const float4 *>(walls)[linedef];
        float dx = ends.z - ends.x, dy = ends.w - ends.y;
        if (kind < 0 || kind >= 20) { dx = -dx; dy = -dy; }      // the seg runs backwards on sidedef 1
        float turn = fmodf(atan2f(dy, dx), TWO_PI);
        if (turn != 0.0f && turn < 0.0f) turn += TWO_PI;         // torch.remainder with a positive divisor
        const i64 fine = (i64)floorf(turn * FINE_PER_RADIAN) & (FINE_ANGLES - 1);
        int32_t *state = decal_state + (lane + place) * 3;
        state[0] = (int32_t)linedef; state[1] = (int32_t)kind; state[2] = own >= 0 ? 1 : 0;
        float *geom = decal_geom + (lane + place) * 4;
        geom[0] = along[lane + s]; geom[1] = impact_z[lane + s];
        geom[2] = (float)fine_sine[(fine + FINE_ANGLES / 4) & (FINE_ANGLES - 1)] / 65536.0f; geom[3] = (float)fine_sine[fine] / 65536.0f;
    }
}

// gd_pack_hud: one thread per lane (engine.py:15209-15262).  As Torch operators these are some forty kernels, which the host takes 0.33 ms to
// launch: as much as all else of a small batch's frame.
__global__ void __launch_bounds__(64) pack_hud_kernel(gd_hud_desc d) {
    const int lane = blockIdx.x * blockDim.x + threadIdx.x;
    if (lane >= d.lane_count) return;
    const auto word = [&](const int64_t *words, int k) -> i64 { return (d.narrow >> k) & 1 ? reinterpret_cast<const int32_t *>(words)[lane] : words[lane]; };
    const auto shown = [](float v) -> i64 { return (i64)(v < 0.0f ? 0.0f : (v > 999.0f ? 999.0f : v)); };      // clamp keeps what is not a number
    const i64 health = shown(d.health[lane]), armor = shown(d.armor[lane]);
    const i64 hurt = 100 - health, twentieth = hurt >= 0 ? hurt / 20 : -((19 - hurt) / 20), pain = clampi(twentieth, 0, 4);
    i64 face = 13 + pain * 3 + word(d.mugshot_face_index, 0);
    if (word(d.attack_held_tics, 4) >= 70) face = 49 + pain;                       // engine.py:175 (70 tics of fire to a rampage)
    if (word(d.mugshot_pain_tics, 2) > 0) face = d.mugshot_ouch[lane] ? 59 + pain : 44 + 5 * word(d.mugshot_pain_direction, 3) + pain;
    if (word(d.mugshot_grin_tics, 1) > 0) face = 64 + pain;
    if (health <= 0) face = 69;
    int owned = 0;
    for (int weapon = 0; weapon < 5; ++weapon) owned |= (d.weapons[(size_t)lane * d.weapon_columns + weapon + 1] != 0.0f ? 1 : 0) << weapon;
    int32_t *out = d.hud_state + (size_t)lane * 9;
    out[0] = (int32_t)(i64)(d.ammo_slot[lane] < 0 ? 0.0f : d.hud_ready_ammo[lane]);
    out[1] = (int32_t)health; out[2] = (int32_t)armor; out[3] = (int32_t)face; out[4] = owned;
    for (int k = 0; k < 4; ++k) out[5 + k] = (int32_t)(i64)d.hud_ammo_counts[(size_t)lane * d.ammo_columns + k];
}

// gd_screen_blend: one thread per lane.  Torch divides by a constant on the device by multiplying with its reciprocal.
__global__ void __launch_bounds__(256) screen_blend_kernel(const int64_t *bonus_count, const int64_t *damage_count, const float *damage_to_alpha, int lane_count, float *blend) {
    const int lane = blockIdx.x * blockDim.x + threadIdx.x;
    if (lane >= lane_count) return;
    const float per = 1.0f / 255.0f, bonus = (float)bonus_count[lane] * 8.0f;
    blend[2 * (size_t)lane] = (bonus < 128.0f ? bonus : 128.0f) * per;
    blend[2 * (size_t)lane + 1] = damage_to_alpha[clampi(damage_count[lane], 0, 113)] * per;
}

#define HIP_TRY GD_HIP_TRY
#define SIZE_CHECK GD_SIZE_CHECK

}  // namespace

// Every kernel of a frame runs on the caller's stream.  (Cutting a batch into chunks or halves pipelined over
// more streams measured no faster: the kernels already fill the machine.)
struct gd_renderer {
    int device;                              // where everything below lies
    DeviceMap dm;
    Scratch sc;
    int chunk_lanes;
    int assembly;                            // GD_ASSEMBLY_*: how frames are put together after the walls (see launch_chunk)
    unsigned char *scratch_block;            // the one allocation `sc` is laid out in (null for a renderer made for 0 lanes)
    size_t scratch_bytes;
    std::vector<void *> allocations;
    hipEvent_t events[16];
    bool events_ready;
    // The flat pass (short kernels that leave most of the chip idle) runs beside the plane shading on a stream of the
    // renderer's own: forked from the caller's stream after the walls, joined before the billboards.
    hipStream_t side_stream;
    hipEvent_t fork_event, join_event;
    bool side_ready;
    // gd_renderer_mark_status: is the next gd_render call to say where its frames' status bits are final; did the last one, and on which stream?
    hipEvent_t status_event;
    bool status_wanted, status_marked;
    hipStream_t status_stream;
    Overlays overlays;                       // device pointers, counts 0 until gd_renderer_set_overlays
    std::vector<void *> overlay_allocations;
};

namespace {

// A renderer's device as the current one, for a call that does not launch on a caller's stream.
struct OnDevice {
    int before = -1;
    hipError_t error;
    explicit OnDevice(int device) {
        error = hipGetDevice(&before);
        if (error == hipSuccess && before != device) error = hipSetDevice(device);
        else before = -1;
    }
    ~OnDevice() { if (before >= 0) (void)hipSetDevice(before); }
};

// Working memory of callers that may not allocate (gd_render_static): one array per device, held until the
// process ends; 23 lanes of a 4000-linedef map of 400 sectors.  (A batch lasts as long as its longest strips, so a chunk more costs the
// time of a small batch: 16 such lanes 0.55 ms in one chunk, 0.97 ms in the two that 64 MiB make of them.)  In host code the array's name only stands for the symbol; its address on the current
// device comes from hipGetSymbolAddress, once per device.
#define STATIC_SCRATCH_BYTES ((size_t)GD_STATIC_SCRATCH_MIB << 20)
#define STATIC_SCRATCH_DEVICES 64
}  // namespace
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];
namespace {
unsigned char *g_static_scratch[STATIC_SCRATCH_DEVICES];

int static_scratch_address(unsigned char **out) {
    int device = 0;
    HIP_TRY(hipGetDevice(&device));
    if (device < 0 || device >= STATIC_SCRATCH_DEVICES) return fail(GD_E_ARG, "device ordinal beyond the static working memory table");
    if (!g_static_scratch[device]) {
        unsigned char *ptr = nullptr;
        HIP_TRY(hipGetSymbolAddress(reinterpret_cast<void **>(&ptr), HIP_SYMBOL(scratch)));
        if (!ptr) return fail(GD_E_HIP, "hipGetSymbolAddress returned no address for the static working memory");
        g_static_scratch[device] = ptr;
    }
    if (out) *out = g_static_scratch[device];
    return GD_OK;
}

// ---------------------------------------------------------------------------------------------
// the float32 inputs the reference evaluates with Torch (gd_ray_tables, gd_sprite_depth)
// ---------------------------------------------------------------------------------------------
// One kernel each for what is seventeen Torch kernels (each a launch of 2-3 us on the device, 5-10 us on the host) otherwise:
// the two together take 0.01 ms at 4096 lanes with 128 billboards, where the Torch operators took 0.1 ms, and a small call
// no longer waits for their launches.  Every operation is rounded on its own, in the operators' order; cosf, sinf, atan2f and
// fmodf are the device library's, which the Torch kernels call as well: equal on every float32 bit pattern.
__device__ __forceinline__ void ray_of(const float *angle, const float *offsets, int k, float *ray_cos, float *ray_sin) {
    const int n = k / SW;
    const float ray = angle[n] + offsets[k - n * SW];
    ray_cos[k] = cosf(ray);
    ray_sin[k] = sinf(ray);
}
__global__ void __launch_bounds__(256) ray_tables_kernel(const float *angle, const float *offsets, int total, float *ray_cos, float *ray_sin) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < total) ray_of(angle, offsets, k, ray_cos, ray_sin);
}

__device__ __forceinline__ void depth_of(const float *x, const float *y, const float *angle, const float *sprite_x, const float *sprite_y, long long k, int slots, float *depth) {
    const int n = (int)(k / slots);
    const float PI = (float)3.14159265358979323846, TWO_PI = (float)(2.0 * 3.14159265358979323846);
    const float dx = sprite_x[k] - x[n], dy = sprite_y[k] - y[n];
    float distance = sqrtf(dx * dx + dy * dy);
    distance = distance < 1.0f ? 1.0f : distance;   // clamp_min keeps what is not a number
    float turn = fmodf((atan2f(dy, dx) - angle[n]) + PI, TWO_PI);
    if (turn != 0.0f && turn < 0.0f) turn += TWO_PI;   // torch.remainder with a positive divisor
    depth[k] = distance * cosf(turn - PI);
}
__global__ void __launch_bounds__(256) sprite_depth_kernel(const float *x, const float *y, const float *angle, const float *sprite_x,
                                                           const float *sprite_y, long long total, int slots, float *depth) {
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < total) depth_of(x, y, angle, sprite_x, sprite_y, k, slots, depth);
}
// Both in one launch, the rays' work-groups first: a launch less in front of every frame with billboards.  (The host's share of the descriptors 37 -> 29 us;
// a view of one lane, 285 us, and 48 RGB frames, 760 us, gain less than two runs of one side differ by.)
__global__ void __launch_bounds__(256) lane_floats_kernel(const float *x, const float *y, const float *angle, const float *offsets, int rays, float *ray_cos, float *ray_sin,
                                                          const float *sprite_x, const float *sprite_y, long long billboards, int slots, float *depth) {
    const unsigned ray_blocks = ((unsigned)rays + 255u) / 256u;
    if (blockIdx.x < ray_blocks) {
        const int k = blockIdx.x * blockDim.x + threadIdx.x;
        if (k < rays) ray_of(angle, offsets, k, ray_cos, ray_sin);
    } else {
        const long long k = (long long)(blockIdx.x - ray_blocks) * blockDim.x + threadIdx.x;
        if (k < billboards) depth_of(x, y, angle, sprite_x, sprite_y, k, slots, depth);
    }
}

__global__ void fill_words_kernel(unsigned int *words, size_t count, unsigned int value) {
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < count; k += (size_t)gridDim.x * blockDim.x) words[k] = value;
}

// Blocks of the spill pool (320 columns each, 641 KiB) for a chunk of `lanes` lanes: every column of up to eight
// lanes, one column in 32 of a large chunk (80 MiB at 4096 lanes).  The static working memory has room for one.
size_t spill_pool_blocks(int lanes) {
    const int share = lanes / 32 > 8 ? lanes / 32 : 8;
    return (size_t)(lanes < share ? lanes : share);
}
#define STATIC_SPILL_BLOCKS 1

// Lay the per-chunk buffers of `sc` out in one block of device memory for `L` lanes of map `h` (every buffer
// 256-byte aligned) and return the bytes the layout takes; with a null `base` nothing is assigned and the call
// only measures.  `status` is not part of the block: the renderer keeps it.  `depth`: also the scene depth plane
// of frames that draw decals; `fused`: also the texels of masked mid-textures that are put together in LDS.
size_t carve_scratch(Scratch &sc, unsigned char *base, size_t L, const gd_map_desc &h, int masked_count, bool depth, bool fused, size_t spill_blocks) {
    size_t used = 0;
    auto take = [&](auto **field, size_t count) {
        typedef typename std::remove_reference<decltype(**field)>::type T;
        used = (used + 255) & ~(size_t)255;
        if (base) *field = reinterpret_cast<T *>(base + used);
        used += (count ? count : 1) * sizeof(T);
    };
    const size_t W = h.wall_count, PX = (size_t)VH * SW, levels = (size_t)(h.floor_level_count + h.ceil_level_count);
    take(&sc.ctx, L);
    take(&sc.rec, L * W);
    take(&sc.span, L * W);
    take(&sc.geo, L * W);
    take(&sc.geo_slot, L * W);
    take(&sc.named, L * ((W + 31) / 32));
    take(&sc.own_rows, L);
    sc.lane_stride = (int)L;
    take(&sc.masked_geo, L * (size_t)masked_count);
    take(&sc.masked_hit, L * SW);
    take(&sc.frag_rec, L * (size_t)(h.split_count > 0 ? h.split_count * h.fragment_slots : 1));
    take(&sc.cand, L * CAND_MAX * SW + spill_blocks * SPILL_DEPTH * SW);   // byte offsets into it are 32 bits wide: L <= 4096, spill_blocks <= 512
    sc.spill_base = (unsigned)(L * CAND_MAX * SW); sc.spill_slots = (int)(spill_blocks * SW);
    take(&sc.cand_count, L * SW);
    take(&sc.spill_columns, spill_blocks * SW);
    take(&sc.spill_count, 1);
    take(&sc.flat_sector, L * PX);
    take(&sc.flat_flags, L * PX);
    take(&sc.flat_span, L * 4);
    take(&sc.flat_tail, L * 2 * SW);
    take(&sc.flat_spans, L * 2);
    take(&sc.flat_span_count, 1);
    take(&sc.flat_rows, L * (size_t)VH);
    take(&sc.flat_row_count, 2);
    take(&sc.gap_columns, L * SW);
    take(&sc.gap_column_count, 1);
    sc.pass_slots = h.sector_count < 16 ? 16 : (h.sector_count > PASS_MAX ? PASS_MAX : h.sector_count);
    take(&sc.pass_rec, L * (size_t)sc.pass_slots * SW);
    take(&sc.pass_path_distance, L * (size_t)sc.pass_slots * SW);
    take(&sc.pass_rows, L * (size_t)sc.pass_slots * SW);
    take(&sc.pass_count, L * SW);
    take(&sc.meta, L * PX);
    if (fused && masked_count > 0) take(&sc.masked_texel, L * PX);
    take(&sc.level_reach, L * levels);
    take(&sc.level_far, L * levels);
    take(&sc.level_masks, L * LEVEL_BUCKETS * (size_t)(levels <= 32 * LEVEL_MASK_WORDS_MAX ? (levels + 31) / 32 : 1));
    take(&sc.level_plane, L * levels * 2);
    take(&sc.row_slope, L * (size_t)VH);
    take(&sc.step_scale, L * STEP_TABLE);
    take(&sc.block_hit, L * SW);
    take(&sc.sprite_listed, L);
    take(&sc.lane_blends, L);
    take(&sc.strip_key, L * SEGS_PER_LANE);
    take(&sc.strip_order, L * SEGS_PER_LANE);
    static_assert((SW / SPRITE_COLUMNS) * SPRITE_ROW_PARTS <= SEGS_PER_LANE * (int)sizeof(int), "Scratch::sprite_late: a byte a work-group");
    sc.sprite_late = reinterpret_cast<unsigned char *>(sc.strip_order);
    if (depth) take(&sc.scene_depth, L * PX);
    take(&sc.frame, L * (size_t)GD_SCREEN_HEIGHT * SW);   // where a frame is put together kernel by kernel when the caller takes none
    return (used + 255) & ~(size_t)255;
}

template <typename T>
int upload(gd_renderer *r, const T *host, size_t count, const T **device) {
    if (count == 0) count = 1;
    void *ptr = nullptr;
    HIP_TRY(hipMalloc(&ptr, count * sizeof(T)));
    r->allocations.push_back(ptr);
    if (host) HIP_TRY(hipMemcpy(ptr, host, count * sizeof(T), hipMemcpyHostToDevice));
    else HIP_TRY(hipMemset(ptr, 0, count * sizeof(T)));
    *device = static_cast<const T *>(ptr);
    return GD_OK;
}

template <typename T>
int scratch_alloc(gd_renderer *r, size_t count, T **device) {
    void *ptr = nullptr;
    HIP_TRY(hipMalloc(&ptr, (count ? count : 1) * sizeof(T)));
    r->allocations.push_back(ptr);
    *device = static_cast<T *>(ptr);
    return GD_OK;
}

// Bounding boxes of the sectors, grouped by plane level (floors first).  The box of a sector is
// that of its edges padded by half a map unit; the even-odd test of engine.py:9598-9617 counts
// edges to the right of the point, so a sector whose boundary is not a set of closed loops can
// also test inside anywhere to the left of its edges and its box is open on that side.
void build_level_boxes(const gd_map_desc *h, std::vector<int> &ofs, std::vector<float4> &boxes) {
    const int S = h->sector_count;
    std::vector<float4> sector_box(S);
    std::vector<char> has_box(S, 0);
    for (int s = 0; s < S; ++s) {
        float x0 = GD_INF, y0 = GD_INF, x1 = -GD_INF, y1 = -GD_INF;
        std::map<std::pair<float, float>, int> degree;
        for (int k = h->sector_edge_ofs[s]; k < h->sector_edge_ofs[s + 1]; ++k) {
            const float *w = h->walls + 4 * h->sector_edge_idx[k];
            for (int e = 0; e < 2; ++e) {
                float x = w[2 * e] + 0.0f, y = w[2 * e + 1] + 0.0f;
                x0 = std::fmin(x0, x); x1 = std::fmax(x1, x); y0 = std::fmin(y0, y); y1 = std::fmax(y1, y);
                ++degree[std::make_pair(x, y)];
            }
            has_box[s] = 1;
        }
        bool closed = true;
        for (const auto &entry : degree) closed = closed && (entry.second % 2 == 0);
        if (!closed) x0 = -GD_INF;
        sector_box[s] = make_float4(x0 - 0.5f, y0 - 0.5f, x1 + 0.5f, y1 + 0.5f);
    }
    ofs.assign(1, 0);
    for (int side = 0; side < 2; ++side) {
        const float *levels = side == 0 ? h->floor_levels : h->ceil_levels;
        const int count = side == 0 ? h->floor_level_count : h->ceil_level_count;
        for (int l = 0; l < count; ++l) {
            for (int s = 0; s < S; ++s)
                if (has_box[s] && h->sector_heights[2 * s + side] == levels[l]) boxes.push_back(sector_box[s]);
            ofs.push_back((int)boxes.size());
        }
    }
}

void build_fine_tables(std::vector<i64> &sine, std::vector<i64> &tangent) {
    // engine.py:309-328
    const double PI = 3.14159265358979323846;
    sine.assign(FINE_ANGLES, 0);
    tangent.assign(FINE_ANGLES / 2, 0);
    const int quarter = FINE_ANGLES / 4;
    for (int i = 0; i < quarter; ++i) sine[i] = (i64)std::trunc(std::sin((double)i * (2.0 * PI / FINE_ANGLES)) * 65536.0);
    for (int i = 0; i < quarter; ++i) sine[quarter + i] = sine[quarter - 1 - i];
    for (int i = 0; i < 2 * quarter; ++i) sine[2 * quarter + i] = -sine[i];
    sine[quarter] = 65536;
    sine[3 * quarter] = -65536;
    for (int i = 0; i < FINE_ANGLES / 2; ++i) {
        double phase = ((double)i - FINE_ANGLES / 4) * (2.0 * PI / FINE_ANGLES);
        if (i == 0) phase += PI / FINE_ANGLES;
        tangent[i] = (i64)std::trunc(std::tan(phase) * 65536.0 + 0.5);
    }
}

// Host-side check of a map descriptor before anything is uploaded: every index a kernel follows must land inside
// its table (a bad one would be a wild device read), and inputs the renderer does not reproduce are refused.
int validate_map(const gd_map_desc *h) {
    const int W = h->wall_count, S = h->sector_count, V = h->vertex_count, T = h->texture_count, K = h->neighbor_slots;
    const void *const needed[] = {h->walls, h->walls_fixed, h->wall_sectors, h->wall_vertex, h->side_tex, h->side_off, h->wall_len,
                                  h->direct_neighbor_table, h->solid_bridge_start_ofs, h->solid_bridge_end_ofs, h->vertex_wall_ofs,
                                  h->sector_wall_ofs, h->sector_edge_ofs, h->grid_cell_ofs, h->grid_item_edge_ofs, h->floor_levels,
                                  h->ceil_levels, h->sector_heights, h->sector_lights, h->sector_floor_tex, h->sector_ceil_tex,
                                  h->tex_atlas, h->tex_w, h->tex_h, h->playpal, h->colormap};
    for (const void *p : needed) if (!p) return fail(GD_E_ARG, "gd_map_desc holds a null table");
    if (V <= 0 || T <= 0 || K < 0 || h->tex_max_h <= 0 || h->tex_max_w <= 0 || h->blocking_count < 0 || h->sprite_count < 0 ||
        h->floor_level_count <= 0 || h->ceil_level_count <= 0 || h->grid_nx <= 0 || h->grid_ny <= 0)
        return fail(GD_E_ARG, "gd_map_desc holds a count out of range");
    if (K > 0 && (!h->endpoint_neighbors || !h->endpoint_neighbor_starts || !h->endpoint_neighbor_ends)) return fail(GD_E_ARG, "missing endpoint neighbour tables");
    if (h->blocking_count > 0 && !h->blocking_walls) return fail(GD_E_ARG, "missing blocking_walls");
    if (h->sprite_count > 0 && (!h->spr_atlas || !h->spr_opaque || !h->spr_post_top || !h->spr_w || !h->spr_h || !h->spr_left || !h->spr_top))
        return fail(GD_E_ARG, "missing sprite patch tables");
    for (int s = 0; s < S; ++s) {
        const float floor_z = h->sector_heights[2 * s], ceiling_z = h->sector_heights[2 * s + 1];
        if (!(floor_z == floor_z) || !(ceiling_z == ceiling_z)) return fail(GD_E_ARG, "sector_heights holds a NaN");
        if (h->sector_floor_tex[s] < 0 || h->sector_floor_tex[s] >= T || h->sector_ceil_tex[s] < 0 || h->sector_ceil_tex[s] >= T)
            return fail(GD_E_ARG, "a sector's flat names a texture out of range");
    }
    for (int t = 0; t < T; ++t)
        if (h->tex_w[t] <= 0 || h->tex_w[t] > h->tex_max_w || h->tex_h[t] <= 0 || h->tex_h[t] > h->tex_max_h || h->tex_w[t] > 32768 || h->tex_h[t] > 32768)
            return fail(GD_E_ARG, "a texture size lies outside 1..32768 or outside the atlas");
    for (int p = 0; p < h->sprite_count; ++p)
        if (h->spr_w[p] < 0 || h->spr_w[p] > h->spr_max_w || h->spr_h[p] < 0 || h->spr_h[p] > h->spr_max_h)
            return fail(GD_E_ARG, "a sprite patch is larger than its atlas");
    for (int w = 0; w < W; ++w) {
        const int front = h->wall_sectors[2 * w], back = h->wall_sectors[2 * w + 1];
        if (front < 0 || front >= S || back < -1 || back >= S) return fail(GD_E_ARG, "wall_sectors names a sector out of range");
        for (int e = 0; e < 2; ++e) if (h->wall_vertex[2 * w + e] < 0 || h->wall_vertex[2 * w + e] >= V) return fail(GD_E_ARG, "wall_vertex names a vertex out of range");
        for (int k = 0; k < 6; ++k) if (h->side_tex[6 * w + k] < -1 || h->side_tex[6 * w + k] >= T) return fail(GD_E_ARG, "side_tex names a texture out of range");
        for (int k = 0; k < K; ++k) if (h->endpoint_neighbors[(size_t)w * K + k] < 0 || h->endpoint_neighbors[(size_t)w * K + k] >= W) return fail(GD_E_ARG, "endpoint_neighbors names a linedef out of range");
        for (int k = 0; k < 2; ++k) if (h->direct_neighbor_table[4 * w + k] < 0 || h->direct_neighbor_table[4 * w + k] >= W) return fail(GD_E_ARG, "direct_neighbor_table names a linedef out of range");
    }
    struct Csr { const int *ofs, *idx; int rows, limit; const char *name; };
    const Csr lists[] = {{h->solid_bridge_start_ofs, h->solid_bridge_start_idx, W, W, "solid_bridge_start"}, {h->solid_bridge_end_ofs, h->solid_bridge_end_idx, W, W, "solid_bridge_end"},
                         {h->vertex_wall_ofs, h->vertex_wall_idx, V, W, "vertex_wall"}, {h->sector_wall_ofs, h->sector_wall_idx, S, W, "sector_wall"},
                         {h->sector_edge_ofs, h->sector_edge_idx, S, W, "sector_edge"}};
    for (const Csr &c : lists) {
        if (c.ofs[0] != 0) return fail(GD_E_ARG, std::string(c.name) + "_ofs must start at 0");
        for (int r = 0; r < c.rows; ++r) if (c.ofs[r + 1] < c.ofs[r]) return fail(GD_E_ARG, std::string(c.name) + "_ofs must not decrease");
        if (c.ofs[c.rows] > 0 && !c.idx) return fail(GD_E_ARG, std::string(c.name) + "_idx is missing");
        for (int k = 0; k < c.ofs[c.rows]; ++k) if (c.idx[k] < 0 || c.idx[k] >= c.limit) return fail(GD_E_ARG, std::string(c.name) + "_idx names a linedef out of range");
    }
    const size_t cells = (size_t)h->grid_nx * h->grid_ny;
    if (h->grid_cell_ofs[0] != 0) return fail(GD_E_ARG, "grid_cell_ofs must start at 0");
    for (size_t c = 0; c < cells; ++c) if (h->grid_cell_ofs[c + 1] < h->grid_cell_ofs[c]) return fail(GD_E_ARG, "grid_cell_ofs must not decrease");
    const int items = h->grid_cell_ofs[cells];
    if (items > 0 && (!h->grid_item_sector || (h->grid_item_edge_ofs[items] > 0 && !h->grid_item_edges))) return fail(GD_E_ARG, "missing grid item tables");
    if (h->grid_item_edge_ofs[0] != 0) return fail(GD_E_ARG, "grid_item_edge_ofs must start at 0");
    for (int it = 0; it < items; ++it) if (h->grid_item_edge_ofs[it + 1] < h->grid_item_edge_ofs[it]) return fail(GD_E_ARG, "grid_item_edge_ofs must not decrease");
    const size_t fine_cells = (size_t)h->fine_nx * h->fine_ny;
    for (size_t k = 0; k < fine_cells; ++k)
        if (FINE_KIND(h->fine_sector[k]) == FINE_DECIDED && (int)(h->fine_sector[k] & 0xFFFFu) >= S) return fail(GD_E_ARG, "fine_sector names a sector out of range");
    return GD_OK;
}

const int STAGE_COUNT = 9;

int launch_chunk(gd_renderer *r, const Scratch &chunk_scratch, const gd_lanes_desc *lanes, const gd_frame_out *out, int base, int count, hipStream_t stream, bool timed, bool mark_status = false) {
    const gd_map_desc &m = r->dm.d;
    Scratch sc = chunk_scratch;
    if (out->final_frames && !out->frames) return fail(GD_E_ARG, "final_frames needs frames");
    if (out->final_frames_layout != GD_LAYOUT_CHW && out->final_frames_layout != GD_LAYOUT_HWC) return fail(GD_E_ARG, "unknown final_frames_layout");
    const size_t frame_stride = (size_t)GD_SCREEN_HEIGHT * SW;
    const size_t F = (size_t)GD_OBS_SIZE * GD_OBS_SIZE;
    const int source_rows = out->obs_source_rows == GD_SCREEN_HEIGHT ? GD_SCREEN_HEIGHT : VH;
    int stage = 0;
    auto mark = [&]() { if (timed) (void)hipEventRecord(r->events[stage], stream); ++stage; };
    // After the walls and the flat selection a frame is put together in one of two ways.  Kernel by kernel through a
    // 320x240 frame in device memory (shade, paint the flat pass's pixels, decals, billboards, overlays, then pool the
    // observation from it), the caller's `indexed` or the working memory's own: the faster way on this chip (its kernels
    // run at full occupancy), and the only one for frames that draw wall decals, which need a per-pixel scene depth.  Or
    // band by band in LDS (band_finish_kernel), the frame never reaching device memory: a fifth less traffic in the
    // assembly for a caller that only wants observations, at five sixths of the speed; chosen with gd_renderer_set_assembly.
    const bool decals = lanes->decal_slots > 0 && lanes->decal_state && lanes->decal_geom && r->overlays.d.decal_variant_count > 0;
    if (!decals) sc.scene_depth = nullptr;
    if (decals && (!sc.scene_depth || !sc.frame)) return fail(GD_E_ARG, "decal working memory missing");
    const bool fused = !decals && (r->assembly == GD_ASSEMBLY_FUSED || (r->assembly == GD_ASSEMBLY_AUTO && !out->indexed && !sc.frame));
    if (fused && r->dm.masked_count > 0 && !sc.masked_texel) return fail(GD_E_ARG, "masked mid-texture working memory missing");
    unsigned char *frame_base = nullptr;
    if (!fused) {
        frame_base = out->indexed ? out->indexed + (size_t)base * frame_stride : sc.frame;
        if (!frame_base) return fail(GD_E_ARG, "assembling the frame kernel by kernel needs an indexed output");
    }
    const bool has_billboards = lanes->sprite_slots > 0 && lanes->sprite_x;
    auto list_billboards = [&](hipStream_t on) { hipLaunchKernelGGL(sprite_list_kernel, dim3(count), dim3(LIST_THREADS), 0, on, r->dm, *lanes, base, count, sc); };
    const bool aside = r->side_ready && side_stream_pays(count, has_billboards);
    mark();
    hipLaunchKernelGGL(lane_tables_kernel, dim3(count), dim3(256), 0, stream, r->dm, *lanes, base, count, sc);
    const bool whole_lanes = setup_whole_lanes(count, m.wall_count);
    if (whole_lanes) hipLaunchKernelGGL(wall_setup_kernel<true>, dim3(1, count), dim3(SETUP_WHOLE_THREADS), 0, stream, r->dm, count, sc);
    else hipLaunchKernelGGL(wall_setup_kernel<false>, dim3((m.wall_count + SETUP_THREADS - 1) / SETUP_THREADS, count), dim3(SETUP_THREADS), 0, stream, r->dm, count, sc);
    if (m.split_count > 0)
        hipLaunchKernelGGL(fragment_setup_kernel, dim3((m.split_count * m.fragment_slots + 63) / 64, count), dim3(64), 0, stream, r->dm, count, sc);
    if (!whole_lanes) hipLaunchKernelGGL(strip_key_kernel, dim3((count * (SW / 64) + 3) / 4), dim3(256), 0, stream, count, sc);
    const int spill_blocks = (sc.spill_slots + 15) / 16;
    hipLaunchKernelGGL(strip_order_kernel, dim3(1 + (spill_blocks < SPILL_BLOCKS ? spill_blocks : SPILL_BLOCKS)), dim3(1024), 0, stream, r->dm, count * SEGS_PER_LANE, sc);
    mark();
    {
        const int wavefronts = (count * SEGS_PER_LANE + 64 / SEG_COLS - 1) / (64 / SEG_COLS);
        const bool split = m.split_count > 0;
        // The longest strips' wavefronts and the others': in one launch, by turns, or the former here and the others on the side stream, both at
        // once (select_together).  This way round: the side stream starts a few microseconds behind, time enough for the longest
        // strips' work-groups to be placed; started together, the other launch's 20,000 take every wavefront slot first and the strips that
        // decide how long the pair lasts begin last.
        const int strips = count * SEGS_PER_LANE;
        const int longest_wanted = select_strips(count, m.wall_count);
        const int longest = strips < longest_wanted ? strips : longest_wanted, others = strips - longest;
        auto pick_select = [&](auto lanes) { constexpr int L = decltype(lanes)::value; return split ? wall_select_kernel<true, L> : wall_select_kernel<false, L>; };
        const int column_lanes = longest > 0 ? select_lanes(count, m.wall_count) : 1;
        auto longest_kernel = column_lanes == 32 ? pick_select(std::integral_constant<int, 32>())
                              : (column_lanes == 16 ? pick_select(std::integral_constant<int, 16>()) : (column_lanes == 8 ? pick_select(std::integral_constant<int, 8>()) : pick_select(std::integral_constant<int, 1>())));
        if (longest == 0 || others == 0 || select_together(count) || !r->side_ready) {
            hipLaunchKernelGGL(longest_kernel, dim3(longest * column_lanes + others), dim3(64), 0, stream, r->dm, sc, 0, longest);
        } else {
            HIP_TRY(hipEventRecord(r->fork_event, stream));
            HIP_TRY(hipStreamWaitEvent(r->side_stream, r->fork_event, 0));
            hipLaunchKernelGGL(longest_kernel, dim3(longest * column_lanes), dim3(64), 0, stream, r->dm, sc, 0, longest);
            hipLaunchKernelGGL(pick_select(std::integral_constant<int, 1>()), dim3(others), dim3(64), 0, r->side_stream, r->dm, sc, longest, 0);
            HIP_TRY(hipEventRecord(r->join_event, r->side_stream));
            HIP_TRY(hipStreamWaitEvent(stream, r->join_event, 0));
        }
        // no kernel behind the selection sets a status bit
        if (mark_status) {
            hipStreamCaptureStatus capturing;
            HIP_TRY(hipStreamIsCapturing(stream, &capturing));
            if (capturing == hipStreamCaptureStatusNone) {      // an event of a capture cannot be waited for
                HIP_TRY(hipEventRecord(r->status_event, stream));
                r->status_marked = true; r->status_stream = stream;
            }
        }
        // the billboards' lists beside the walls' drawing, on the side stream (when stages are being timed, with the billboards)
        if (has_billboards && !fused && !timed) {
            if (aside) {
                HIP_TRY(hipEventRecord(r->fork_event, stream));
                HIP_TRY(hipStreamWaitEvent(r->side_stream, r->fork_event, 0));
            }
            list_billboards(aside ? r->side_stream : stream);
        }
        mark();
        hipLaunchKernelGGL(split ? wall_geometry_kernel<true> : wall_geometry_kernel<false>, dim3(geometry_parts(count) + SW / 64, count), dim3(64), 0, stream, r->dm, count, sc, geometry_parts(count));
        const int parts = raster_sixteen(count) ? 16 : raster_parts(count);
        const dim3 grid((wavefronts * parts + WALL_STRIPS_PER_GROUP - 1) / WALL_STRIPS_PER_GROUP), block(64 * WALL_STRIPS_PER_GROUP);
        const bool general = split || m.sector_count > LDS_SECTORS || m.texture_count > LDS_TEXTURES;
        auto pick = [&](auto parts) {
            constexpr int P = decltype(parts)::value;
            return decals ? (general ? wall_raster_kernel<true, true, P> : wall_raster_kernel<true, false, P>)
                          : (general ? wall_raster_kernel<false, true, P> : wall_raster_kernel<false, false, P>);
        };
        auto kernel = parts == 16 ? pick(std::integral_constant<int, 16>()) : parts == 8 ? pick(std::integral_constant<int, 8>()) : parts == 4 ? pick(std::integral_constant<int, 4>())
                      : parts == 2 ? pick(std::integral_constant<int, 2>()) : pick(std::integral_constant<int, 1>());
        hipLaunchKernelGGL(kernel, grid, block, 0, stream, r->dm, count, sc, frame_base, frame_stride);
    }
    mark();
    // The plane shading and the flat pass do not depend on each other: the first reads the per-pixel words and writes the
    // pixels some drawseg owns, the second reads the same words and writes its own planes and, at the end, the pixels no
    // drawseg owns.  The flat pass is a chain of short kernels that wait more than they compute; it stays on the
    // caller's stream, where its first kernel starts the moment the traversal ends, and the shading goes to the renderer's
    // side stream, a few microseconds behind (the other way round the shading takes every compute unit before the first
    // block of the flat pass is placed).  (Not when stages are being timed.)
    const bool beside = !fused && !timed && aside;
    hipStream_t shade_stream = stream;
    if (beside) {
        HIP_TRY(hipEventRecord(r->fork_event, stream));
        HIP_TRY(hipStreamWaitEvent(r->side_stream, r->fork_event, 0));
        shade_stream = r->side_stream;
    }
    // timed (and so serial): shading, then the flat pass, each between its own marks
    auto shade_planes = [&]() {
        if (fused) return;
        hipLaunchKernelGGL(plane_shade_kernel, dim3((SHADE_TILES + SHADE_THREADS / 64 - 1) / (SHADE_THREADS / 64), count), dim3(SHADE_THREADS), 0, shade_stream, r->dm, count, sc, frame_base, frame_stride);
    };
    if (!beside) shade_planes();
    mark();
    // the flat pass, where the walls left it something to decide
    // The sizes of its work lists are known on the device only: each kernel's grid follows the lanes, a block takes one entry after another.
    auto flat_grid = [count](int per_lane, int most) { return dim3((unsigned)(count >= most / per_lane ? most : (count * per_lane < 32 ? 32 : count * per_lane))); };
    const int plane_levels = m.floor_level_count + m.ceil_level_count;
    const bool level_masks = plane_levels > LEVEL_MASK_MIN_LEVELS && plane_levels <= 32 * LEVEL_MASK_WORDS_MAX;   // level_mask_words() > 0
    const int waves = gap_waves(count, m.wall_count);
    hipLaunchKernelGGL(waves == 16 ? flat_gap_kernel<16> : (waves == 8 ? flat_gap_kernel<8> : flat_gap_kernel<4>), flat_grid(8, 16384 / waves), dim3(64 * waves), 0, stream,
                       r->dm, *lanes, base, sc);
    hipLaunchKernelGGL(flat_rows_kernel, dim3((count + ROWS_LANES - 1) / ROWS_LANES), dim3(64 * ROWS_LANES), 0, stream, count, sc);
    hipLaunchKernelGGL(level_masks ? flat_span_select_kernel<true> : flat_span_select_kernel<false>, flat_grid(16, 2048), dim3(256), 0, stream, r->dm, *lanes, base, sc);
    mark();
    hipLaunchKernelGGL(level_masks ? flat_tail_kernel<true> : flat_tail_kernel<false>, flat_grid(16, 2048), dim3(256), 0, stream, r->dm, *lanes, base, count, sc);
    hipLaunchKernelGGL(flat_span_finish_kernel, flat_grid(2, 1024), dim3(FINISH_THREADS), 0, stream, sc);
    // Billboards need not wait for the flat pass's pixels, but where one blends with such a pixel (sprite_style): they are painted right after the
    // shading, on the side stream, and mark the gap pixels they take; the flat pass's pixels are painted after the join, around the marks, and the
    // few that are blended with after these.  The flat chain, which waits for memory most of its time, then has the billboards beside it
    // as well as the shading.  (When the lanes with any billboard that blends waited with all of theirs: 1024 lanes on the 2000-linedef map, a
    // quarter of them so, 1094 us; now 1050.)  In frames with decals, which go between the flat pass and the billboards, all wait: to paint
    // early what covers, and to mark it for the decals, leaves so much to the late launch that 2048 lanes take 2146 us instead of 2102.
    const bool billboards_split = beside && has_billboards && !decals;
    const bool left_over = billboards_split && lanes->sprite_style != nullptr;   // may the early launch leave pixels?
    auto paint_billboards = [&](hipStream_t on, int phase) {
        const bool blends = lanes->sprite_style != nullptr;
        auto kernel = phase == SPRITES_LATE ? sprite_pixels_kernel<SPRITES_LATE, true>
                      : phase == SPRITES_EARLY ? (blends ? sprite_pixels_kernel<SPRITES_EARLY, true> : sprite_pixels_kernel<SPRITES_EARLY, false>)
                                               : (blends ? sprite_pixels_kernel<SPRITES_ALL, true> : sprite_pixels_kernel<SPRITES_ALL, false>);
        hipLaunchKernelGGL(kernel, dim3(SW / SPRITE_COLUMNS, count, sprite_row_parts(count)), dim3(SPRITE_THREADS), 0, on, r->dm, *lanes, base, count, sc, frame_base, frame_stride);
    };
    auto shade_gaps = [&]() { hipLaunchKernelGGL(flat_shade_kernel, flat_grid(4, 4096), dim3(64), 0, stream, r->dm, sc, frame_base, frame_stride); };
    if (!fused && !billboards_split) shade_gaps();
    if (beside) {
        shade_planes();
        if (billboards_split) paint_billboards(r->side_stream, SPRITES_EARLY);
        HIP_TRY(hipEventRecord(r->join_event, r->side_stream));
        HIP_TRY(hipStreamWaitEvent(stream, r->join_event, 0));
        if (billboards_split) shade_gaps();
    }
    mark();
    const float *blend = lanes->screen_blend ? lanes->screen_blend + 2 * (size_t)base : nullptr;
    if (fused) {
        FinishOut finish;
        finish.indexed = out->indexed ? out->indexed + (size_t)base * frame_stride : nullptr;
        finish.rgb = out->rgb ? out->rgb + (size_t)base * frame_stride * 3 : nullptr;
        finish.obs = out->obs ? out->obs + (size_t)base * F : nullptr;
        finish.frames = out->frames ? out->frames + (size_t)base * GD_FRAME_STACK * F : nullptr;
        finish.final_frames = out->final_frames ? out->final_frames + (size_t)base * GD_FRAME_STACK * F : nullptr;
        finish.reset_mask = out->reset_mask ? out->reset_mask + base : nullptr;
        finish.blend = blend;
        finish.stack_mode = out->stack_mode;
        finish.final_hwc = out->final_frames_layout == GD_LAYOUT_HWC;
        finish.source_rows = source_rows;
        const bool sprites = lanes->sprite_slots > 0 && lanes->sprite_x;
        size_t shared = sprites ? (size_t)lanes->sprite_slots * sizeof(SpriteRec) : 0;
        if (shared <= (size_t)LDS_SECTORS * sizeof(float4) + 32 * 256) shared = 0;   // the records reuse the shading tables' LDS
        hipLaunchKernelGGL(band_finish_kernel, dim3(BAND_COUNT, count), dim3(BAND_THREADS), shared, stream, r->dm, r->overlays, *lanes, base, count, sc, finish);
        mark();
        mark();
        HIP_TRY(hipGetLastError());
        return GD_OK;
    }
    if (decals)
        hipLaunchKernelGGL(decal_kernel, dim3(count), dim3(SW), 0, stream, r->dm, r->overlays, *lanes, base, count, sc, frame_base, frame_stride);
    if (has_billboards && timed) list_billboards(stream);
    if (has_billboards && (!billboards_split || left_over)) paint_billboards(stream, billboards_split ? SPRITES_LATE : SPRITES_ALL);
    if (lanes->weapon_state && r->overlays.d.weapon_patch_count > 0)
        hipLaunchKernelGGL(weapon_overlay_kernel, dim3(WEAPON_PARTS, count), dim3(WEAPON_THREADS), 0, stream, r->overlays, lanes->weapon_state, base, count,
                           frame_base, frame_stride);
    if (lanes->hud_state && r->overlays.d.hud_patch_count > 0)
        hipLaunchKernelGGL(hud_kernel, dim3(HUD_TILES / (HUD_THREADS / 64), count), dim3(HUD_THREADS), 0, stream, r->overlays, lanes->hud_state, base, count, frame_base, frame_stride);
    mark();
    if (out->obs || out->frames) {
        launch_observe(stream, frame_base, frame_stride, source_rows, m.playpal, count, out->obs ? out->obs + (size_t)base * F : nullptr,
                       out->frames ? out->frames + (size_t)base * GD_FRAME_STACK * F : nullptr, out->reset_mask ? out->reset_mask + base : nullptr, out->stack_mode,
                       out->final_frames ? out->final_frames + (size_t)base * GD_FRAME_STACK * F : nullptr, out->final_frames_layout == GD_LAYOUT_HWC, blend);
    }
    if (out->rgb) {
        size_t pixels = (size_t)count * frame_stride;
        hipLaunchKernelGGL(expand_rgb_kernel, dim3((unsigned)((pixels + EXPAND_PIXELS - 1) / EXPAND_PIXELS)), dim3(EXPAND_THREADS), 0, stream, frame_base, m.playpal, pixels,
                           out->rgb + (size_t)base * frame_stride * 3, blend, (size_t)GD_SCREEN_HEIGHT * SW);
    }
    mark();
    HIP_TRY(hipGetLastError());
    return GD_OK;
}

}  // namespace

extern "C" {

const char *gd_version(void) { return "gradoom_amd 0.2.0 (gfx950)"; }
uint32_t gd_abi_version(void) { return GD_ABI_VERSION; }
const char *gd_last_error(void) { return g_error.c_str(); }

int gd_renderer_create(const gd_map_desc *h, const float *cosine_correction, int32_t max_lanes, gd_renderer **out) {
    if (!h || !out || !cosine_correction) return fail(GD_E_ARG, "null argument");
    SIZE_CHECK(h, gd_map_desc);
    if (max_lanes < 0) return fail(GD_E_ARG, "max_lanes must not be negative");
    if (h->wall_count <= 0 || h->sector_count <= 0) return fail(GD_E_ARG, "empty map");
    if (h->wall_count >= 65535) return fail(GD_E_ARG, "at most 65534 linedefs");
    if (h->sector_count >= 8191) return fail(GD_E_ARG, "at most 8190 sectors");
    if (h->vertex_count >= 65536) return fail(GD_E_ARG, "at most 65535 distinct vertices");
    if (h->fine_nx <= 0 || h->fine_ny <= 0 || !(h->fine_cell > 0.0f) || !h->fine_sector) return fail(GD_E_ARG, "missing fine point-location raster");
    if (h->grid_cell != 8.0f * h->fine_cell || (h->fine_nx + 7) / 8 > h->grid_nx || (h->fine_ny + 7) / 8 > h->grid_ny)
        return fail(GD_E_ARG, "grid_cell must be 8 * fine_cell and the coarse grid must cover the fine raster");
    if (h->fragment_slots < 1 || h->split_count < 0 || h->split_count > h->wall_count || !h->wall_split_slot ||
        (h->split_count > 0 && (!h->split_fragments_fixed || !h->split_fragment_mask)))
        return fail(GD_E_ARG, "invalid projection fragment tables");
    for (int w = 0; w < h->wall_count; ++w)
        if (h->wall_split_slot[w] < -1 || h->wall_split_slot[w] >= h->split_count)
            return fail(GD_E_ARG, "wall_split_slot names a row outside the fragment tables");
    if (!h->additive_luts || !h->translucent_lut) return fail(GD_E_ARG, "missing sprite blend tables");
    if ((unsigned long long)h->texture_count * (unsigned long long)h->tex_max_h * (unsigned long long)h->tex_max_w >= (1ULL << 32))
        return fail(GD_E_ARG, "the texture atlas must stay below 4 GiB");
    if (int bad = validate_map(h)) return bad;
    gd_renderer *r = new (std::nothrow) gd_renderer();
    if (!r) return fail(GD_E_ARG, "out of host memory");
    r->events_ready = false;
    r->side_ready = false;
    r->scratch_block = nullptr; r->scratch_bytes = 0;
    r->assembly = GD_ASSEMBLY_AUTO;
    std::memset(&r->sc, 0, sizeof(r->sc));
    std::memset(&r->overlays, 0, sizeof(r->overlays));
    r->dm.d = *h;
    r->device = 0;
    gd_map_desc &d = r->dm.d;
    const size_t W = h->wall_count, S = h->sector_count, V = h->vertex_count, K = h->neighbor_slots;
    int rc = hipGetDevice(&r->device) == hipSuccess ? GD_OK : fail(GD_E_HIP, "hipGetDevice");
#define UP(field, count) if (rc == GD_OK) rc = upload(r, h->field, (size_t)(count), &d.field)
    UP(walls, W * 4); UP(walls_fixed, W * 4); UP(wall_sectors, W * 2);
    UP(side_tex, W * 6);
    UP(endpoint_neighbors, W * K); UP(endpoint_neighbor_starts, W * K); UP(endpoint_neighbor_ends, W * K);
    UP(vertex_wall_ofs, V + 1);
    UP(blocking_walls, h->blocking_count);
    // what only the tables made of them below ask for: no kernel
    d.wall_vertex = d.direct_neighbor_table = d.vertex_wall_idx = d.solid_bridge_start_ofs = d.solid_bridge_end_ofs = nullptr;
    d.sector_wall_ofs = d.sector_wall_idx = d.sector_edge_ofs = d.sector_edge_idx = nullptr;
    d.side_off = d.wall_len = nullptr;
    {
        const size_t fragments = (size_t)(h->split_count > 0 ? h->split_count : 1) * h->fragment_slots;
        UP(wall_split_slot, W);
        if (h->split_count > 0) { UP(split_fragments_fixed, fragments * 4); UP(split_fragment_mask, fragments); }
        else { d.split_fragments_fixed = nullptr; d.split_fragment_mask = nullptr; }
    }
    const size_t cells = (size_t)h->grid_nx * h->grid_ny;
    const size_t items = h->grid_cell_ofs[cells];
    UP(grid_cell_ofs, cells + 1); UP(grid_item_sector, items); UP(grid_item_edge_ofs, items + 1);
    UP(grid_item_edges, h->grid_item_edge_ofs[items]);
    UP(fine_sector, (size_t)h->fine_nx * h->fine_ny);
    UP(floor_levels, h->floor_level_count); UP(ceil_levels, h->ceil_level_count);
    UP(sector_heights, S * 2); UP(sector_lights, S); UP(sector_floor_tex, S); UP(sector_ceil_tex, S);
    const size_t texels = (size_t)h->texture_count * h->tex_max_h * h->tex_max_w;
    UP(tex_atlas, texels); UP(tex_w, h->texture_count); UP(tex_h, h->texture_count);
    UP(playpal, 768); UP(colormap, 34 * 256);
    const size_t sprels = (size_t)h->sprite_count * h->spr_max_h * h->spr_max_w;
    UP(spr_atlas, sprels); UP(spr_opaque, sprels); UP(spr_post_top, sprels);
    {
        std::vector<unsigned int> words(sprels);
        for (size_t k = 0; k < sprels; ++k) words[k] = (unsigned)h->spr_atlas[k] | ((unsigned)h->spr_post_top[k] << 8) | (h->spr_opaque[k] ? 1u << 16 : 0u);
        if (rc == GD_OK) rc = upload(r, words.data(), words.size(), &r->dm.sprite_texels);
    }
    UP(spr_w, h->sprite_count); UP(spr_h, h->sprite_count); UP(spr_left, h->sprite_count); UP(spr_top, h->sprite_count);
    UP(additive_luts, 2 * 256 * 256); UP(translucent_lut, 256 * 256);
#undef UP
    std::vector<i64> sine, tangent;
    build_fine_tables(sine, tangent);
    if (rc == GD_OK) rc = upload(r, sine.data(), sine.size(), &r->dm.fine_sine);
    if (rc == GD_OK) rc = upload(r, tangent.data(), tangent.size(), &r->dm.fine_tangent);
    if (rc == GD_OK) rc = upload(r, cosine_correction, (size_t)SW, &r->dm.cosine_correction);
    {
        std::vector<float> inverse(SW);
        for (int x = 0; x < SW; ++x) inverse[x] = 1.0f / cosine_correction[x];   // IEEE division, as on the device
        if (rc == GD_OK) rc = upload(r, inverse.data(), inverse.size(), &r->dm.inverse_cosine);
        for (int strip = 0; strip < SW / 64; ++strip) {
            float smallest = cosine_correction[strip * 64];
            for (int x = strip * 64; x < strip * 64 + 64; ++x) smallest = std::fmin(smallest, cosine_correction[x]);
            r->dm.strip_reach_scale[strip] = smallest > 0.0f ? 1.001f / smallest : GD_INF;
            float largest = cosine_correction[strip * 64];
            for (int x = strip * 64; x < strip * 64 + 64; ++x) largest = std::fmax(largest, cosine_correction[x]);
            r->dm.strip_far_scale[strip] = smallest > 0.0f && std::isfinite(largest) ? 0.999f / largest : 0.0f;
        }
        r->dm.fine_inverse = 1.0f / h->fine_cell;
    }
    {
        std::vector<int> box_ofs;
        std::vector<float4> boxes;
        build_level_boxes(h, box_ofs, boxes);
        if (rc == GD_OK) rc = upload(r, box_ofs.data(), box_ofs.size(), &r->dm.level_box_ofs);
        if (rc == GD_OK) rc = upload(r, boxes.data(), boxes.size(), &r->dm.level_boxes);
        std::vector<float4> around(box_ofs.size() - 1, make_float4(GD_INF, GD_INF, -GD_INF, -GD_INF));   // a level without a sector: no point
        for (size_t l = 0; l + 1 < box_ofs.size(); ++l)
            for (int k = box_ofs[l]; k < box_ofs[l + 1]; ++k) {
                const float4 box = boxes[k];
                around[l] = make_float4(std::fmin(around[l].x, box.x), std::fmin(around[l].y, box.y), std::fmax(around[l].z, box.z), std::fmax(around[l].w, box.w));
            }
        if (rc == GD_OK) rc = upload(r, around.data(), around.size(), &r->dm.level_box);
        std::vector<int> facts(W, 0);
        for (size_t w = 0; w < W; ++w)
            facts[w] = (h->wall_sectors[2 * w + 1] < 0 ? WALL_ONE_SIDED : 0) | (h->wall_split_slot[w] >= 0 ? WALL_SPLIT : 0) | (h->wall_len[w] <= 32.0f ? WALL_SHORT : 0) |
                       (h->wall_sectors[2 * w] == 0 || h->wall_sectors[2 * w + 1] == 0 ? WALL_SECTOR0 : 0);
        for (int b = 0; b < h->blocking_count; ++b) {
            const int w = h->blocking_walls[b];
            if (w < 0 || (size_t)w >= W) { if (rc == GD_OK) rc = fail(GD_E_ARG, "blocking_walls holds a linedef index out of range"); continue; }
            if ((facts[w] >> WALL_BLOCKING_SHIFT) == 0) facts[w] |= (b + 1) << WALL_BLOCKING_SHIFT;   // the first slot wins ties, like the scan it replaces
        }
        if (rc == GD_OK) rc = upload(r, facts.data(), facts.size(), &r->dm.wall_facts);
        // The solid bridges by the first time each linedef comes in its row, which is all that is asked of it: a row then has fewer than 65536 (WallLinks).
        const int *const bridge_ofs[2] = {h->solid_bridge_start_ofs, h->solid_bridge_end_ofs}, *const bridge_idx[2] = {h->solid_bridge_start_idx, h->solid_bridge_end_idx};
        std::vector<int> bridge_first[2], bridges[2];
        for (int end = 0; end < 2; ++end) {
            std::vector<size_t> seen(W, W);
            for (size_t w = 0; w < W; ++w) {
                bridge_first[end].push_back((int)bridges[end].size());
                for (int k = bridge_ofs[end][w]; k < bridge_ofs[end][w + 1]; ++k) {
                    const int b = bridge_idx[end][k];
                    if (seen[b] != w) bridges[end].push_back(b);
                    seen[b] = w;
                }
            }
            bridge_first[end].push_back((int)bridges[end].size());
        }
        if (rc == GD_OK) rc = upload(r, bridges[0].data(), bridges[0].size(), &d.solid_bridge_start_idx);
        if (rc == GD_OK) rc = upload(r, bridges[1].data(), bridges[1].size(), &d.solid_bridge_end_idx);
        std::vector<WallLinks> links(W);
        for (size_t w = 0; w < W; ++w) {
            WallLinks &link = links[w];      // all zero
            link.sectors = ((unsigned)h->wall_sectors[2 * w] & 0xFFFFu) | (unsigned)h->wall_sectors[2 * w + 1] << 16;
            link.vertices = ((unsigned)h->wall_vertex[2 * w] & 0xFFFFu) | (unsigned)h->wall_vertex[2 * w + 1] << 16;
            for (int k = 0; k < 2; ++k) link.neighbour[k] = h->direct_neighbor_table[4 * w + k];
            link.slots = (unsigned)h->direct_neighbor_table[4 * w + 2];
            for (int end = 0; end < 2; ++end) {
                link.solid[end] = bridge_first[end][w];
                link.solid_counts |= (unsigned)(bridge_first[end][w + 1] - link.solid[end]) << (16 * end);
            }
        }
        if (rc == GD_OK) rc = upload(r, links.data(), links.size(), &r->dm.wall_links);
        std::vector<VertexLink> vertex_links(h->vertex_wall_ofs[V]);
        for (size_t k = 0; k < vertex_links.size(); ++k) vertex_links[k] = {h->vertex_wall_idx[k], links[h->vertex_wall_idx[k]].sectors};
        if (rc == GD_OK) rc = upload(r, vertex_links.data(), vertex_links.size(), &r->dm.vertex_links);
        std::vector<WallSide> sides(W * 2);
        std::vector<int> masked_slot(W, -1);
        r->dm.masked_count = 0;
        for (size_t w = 0; w < W; ++w) {
            const float *l = h->walls + 4 * w;
            const bool horizontal = std::fabs(l[3] - l[1]) < 1e-6f, vertical = std::fabs(l[2] - l[0]) < 1e-6f;
            for (int side = 0; side < 2; ++side) {
                WallSide &ws = sides[w * 2 + side];
                std::memset(&ws, 0, sizeof(ws));
                for (int t = 0; t < 3; ++t) ws.tex[t] = h->side_tex[(w * 2 + side) * 3 + t];
                ws.other = (short)h->wall_sectors[2 * w + (side == 0 ? 1 : 0)];
                ws.offset_x = (i64)std::rint(h->side_off[(w * 2 + side) * 2] * 65536.0f);
                ws.offset_y = h->side_off[(w * 2 + side) * 2 + 1];
                ws.contrast = vertical ? 16.0f : (horizontal ? -16.0f : 0.0f);
                ws.repeat = (i64)std::rint(h->wall_len[w] * 65536.0f);
                if (h->wall_sectors[2 * w + 1] >= 0 && ws.tex[0] >= 0 && masked_slot[w] < 0) masked_slot[w] = r->dm.masked_count++;
            }
        }
        if (rc == GD_OK) rc = upload(r, sides.data(), sides.size(), &r->dm.wall_side);
        if (rc == GD_OK) rc = upload(r, masked_slot.data(), masked_slot.size(), &r->dm.masked_slot);
        r->dm.sector_level = nullptr;
        std::vector<unsigned int> pairs(S, 0);
        bool listed = h->floor_level_count <= 65535 && h->ceil_level_count <= 65535;
        if (listed) {
            for (size_t s = 0; s < S; ++s) {
                int fi = -1, ci = -1;
                for (int l = 0; l < h->floor_level_count; ++l) if (h->floor_levels[l] == h->sector_heights[2 * s]) fi = l;
                for (int l = 0; l < h->ceil_level_count; ++l) if (h->ceil_levels[l] == h->sector_heights[2 * s + 1]) ci = l;
                listed = listed && fi >= 0 && ci >= 0;
                pairs[s] = ((unsigned)fi & 0xFFFFu) | (((unsigned)ci & 0xFFFFu) << 16);
            }
            // a sector whose height is missing from the level lists keeps the per-pixel divisions
            if (listed && rc == GD_OK) rc = upload(r, pairs.data(), pairs.size(), &r->dm.sector_level);
        }
        std::vector<int2> cell_range(cells);
        std::vector<int4> cell_item(items);
        std::vector<float4> cell_edge;
        for (size_t c = 0; c < cells; ++c) cell_range[c] = make_int2(h->grid_cell_ofs[c], h->grid_cell_ofs[c + 1]);
        for (size_t it = 0; it < items; ++it) {
            const int entry = h->grid_item_sector[it];
            const size_t s = (size_t)(entry & ~GRID_ALWAYS_INSIDE);
            if (s >= S) { if (rc == GD_OK) rc = fail(GD_E_ARG, "grid_item_sector holds a sector index out of range"); continue; }
            const int first = (int)cell_edge.size();
            for (int k = h->grid_item_edge_ofs[it]; k < h->grid_item_edge_ofs[it + 1]; ++k) {
                const int w = h->grid_item_edges[k];
                if (w < 0 || (size_t)w >= W) { if (rc == GD_OK) rc = fail(GD_E_ARG, "grid_item_edges holds a linedef index out of range"); continue; }
                cell_edge.push_back(make_float4(h->walls[4 * w], h->walls[4 * w + 1], h->walls[4 * w + 2], h->walls[4 * w + 3]));
            }
            // .y: the sector's level indices (as in sector_level), or negative: compare heights (also when the ceiling
            // index would reach the sign bit)
            cell_item[it] = make_int4(entry, listed ? (int)pairs[s] : -1, first, (int)cell_edge.size());
        }
        if (rc == GD_OK) rc = upload(r, cell_range.data(), cell_range.size(), &r->dm.cell_range);
        if (rc == GD_OK) rc = upload(r, cell_item.data(), cell_item.size(), &r->dm.cell_item);
        if (rc == GD_OK) rc = upload(r, cell_edge.data(), cell_edge.size(), &r->dm.cell_edge);
    }
    // Working memory for one chunk of lanes; larger batches are rendered chunk by chunk.  A renderer made for no
    // lanes holds the map only and renders through gd_render_static.
    const int chunk = max_lanes < 4096 ? max_lanes : 4096;
    r->chunk_lanes = chunk;
    Scratch &sc = r->sc;
    if (rc == GD_OK && chunk > 0) {
        unsigned char *block = nullptr;
        const size_t bytes = carve_scratch(sc, nullptr, (size_t)chunk, *h, r->dm.masked_count, false, false, spill_pool_blocks(chunk));
        rc = scratch_alloc(r, bytes, &block);
        if (rc == GD_OK) {
            carve_scratch(sc, block, (size_t)chunk, *h, r->dm.masked_count, false, false, spill_pool_blocks(chunk));
            r->scratch_block = block; r->scratch_bytes = bytes;
        }
    }
    if (rc == GD_OK) {
        // in host memory: whoever has waited for a frame reads them as they are (gd_renderer_status_seen)
        void *words = nullptr;
        if (hipHostMalloc(&words, 64) != hipSuccess) rc = fail(GD_E_HIP, "hipHostMalloc status");
        else { sc.status = static_cast<unsigned char *>(words); sc.status[0] = 0; sc.status[1] = 0; }
    }
    if (rc == GD_OK) rc = static_scratch_address(nullptr);   // looked up once per device, outside any stream capture
    if (rc == GD_OK) {
        for (int i = 0; i < 16; ++i) if (hipEventCreate(&r->events[i]) != hipSuccess) rc = fail(GD_E_HIP, "hipEventCreate");
        r->events_ready = rc == GD_OK;
    }
    if (rc == GD_OK) {
        // default priority, like the caller's stream; no implicit synchronisation with the null stream
        if (hipStreamCreateWithFlags(&r->side_stream, hipStreamNonBlocking) != hipSuccess) rc = fail(GD_E_HIP, "hipStreamCreateWithFlags");
        else if (hipEventCreateWithFlags(&r->fork_event, hipEventDisableTiming) != hipSuccess) { (void)hipStreamDestroy(r->side_stream); rc = fail(GD_E_HIP, "hipEventCreateWithFlags"); }
        else if (hipEventCreateWithFlags(&r->join_event, hipEventDisableTiming) != hipSuccess) {
            (void)hipEventDestroy(r->fork_event); (void)hipStreamDestroy(r->side_stream); rc = fail(GD_E_HIP, "hipEventCreateWithFlags");
        } else r->side_ready = true;
        if (rc == GD_OK && hipEventCreateWithFlags(&r->status_event, hipEventDisableTiming) != hipSuccess) { r->status_event = nullptr; rc = fail(GD_E_HIP, "hipEventCreateWithFlags"); }
    }
    if (rc != GD_OK) { std::string keep = g_error; gd_renderer_destroy(r); g_error = keep; return rc; }
    *out = r;
    return GD_OK;
}

void gd_renderer_destroy(gd_renderer *r) {
    if (!r) return;
    for (void *ptr : r->allocations) (void)hipFree(ptr);
    for (void *ptr : r->overlay_allocations) (void)hipFree(ptr);
    if (r->sc.status) (void)hipHostFree(const_cast<unsigned char *>(r->sc.status));
    if (r->events_ready) for (int i = 0; i < 16; ++i) (void)hipEventDestroy(r->events[i]);
    if (r->side_ready) { (void)hipEventDestroy(r->fork_event); (void)hipEventDestroy(r->join_event); (void)hipStreamDestroy(r->side_stream); }
    if (r->status_event) (void)hipEventDestroy(r->status_event);
    delete r;
}

static int check_render_args(gd_renderer *r, const gd_lanes_desc *lanes, const gd_frame_out *out) {
    if (!r || !lanes || !out) return fail(GD_E_ARG, "null argument");
    SIZE_CHECK(lanes, gd_lanes_desc);
    SIZE_CHECK(out, gd_frame_out);
    if (out->obs_source_rows != 0 && out->obs_source_rows != VH && out->obs_source_rows != GD_SCREEN_HEIGHT)
        return fail(GD_E_ARG, "obs_source_rows must be 208 (or 0) or 240");
    if (lanes->lane_count < 0) return fail(GD_E_ARG, "negative lane count");
    // an empty batch is a call that does nothing: its tensors hold no element and may have no address
    if (lanes->lane_count > 0 && (!lanes->x || !lanes->y || !lanes->angle || !lanes->view_z || !lanes->x_fixed || !lanes->y_fixed ||
                                  !lanes->angle_bam || !lanes->pitch_bam || !lanes->ray_cos || !lanes->ray_sin))
        return fail(GD_E_ARG, "missing lane tensor");
    if (out->stack_mode != GD_STACK_STEP && out->stack_mode != GD_STACK_RESET) return fail(GD_E_ARG, "unknown stack_mode");
    if (lanes->sprite_slots < 0 || lanes->sprite_slots > SPRITE_SLOTS_MAX) return fail(GD_E_ARG, "sprite_slots must be in [0, 512]");
    if (lanes->decal_slots < 0) return fail(GD_E_ARG, "negative decal_slots");
    if (lanes->decal_slots > 0 && (lanes->decal_state != nullptr) != (lanes->decal_geom != nullptr))
        return fail(GD_E_ARG, "decal_state and decal_geom go together");
    if (lanes->sprite_slots > 0 && lanes->sprite_x &&
        (!lanes->sprite_y || !lanes->sprite_z || !lanes->sprite_depth || !lanes->sprite_id || !lanes->sprite_alive))
        return fail(GD_E_ARG, "missing sprite tensor");
    return GD_OK;
}

int gd_render(gd_renderer *r, const gd_lanes_desc *lanes, const gd_frame_out *out, void *stream) {
    int rc = check_render_args(r, lanes, out);
    if (rc != GD_OK) return rc;
    if (r->chunk_lanes <= 0) return fail(GD_E_ARG, "this renderer was created for 0 lanes and holds no working memory: use gd_render_static");
    hipStream_t caller = static_cast<hipStream_t>(stream);
    const bool mark_status = r->status_wanted;
    r->status_wanted = r->status_marked = false;
    for (int base = 0; base < lanes->lane_count; base += r->chunk_lanes) {
        int count = lanes->lane_count - base < r->chunk_lanes ? lanes->lane_count - base : r->chunk_lanes;
        rc = launch_chunk(r, r->sc, lanes, out, base, count, caller, false, mark_status && base + count == lanes->lane_count);
        if (rc != GD_OK) return rc;
    }
    return GD_OK;
}

int gd_render_static(gd_renderer *r, const gd_lanes_desc *lanes, const gd_frame_out *out, void *stream) {
    int rc = check_render_args(r, lanes, out);
    if (rc != GD_OK) return rc;
    unsigned char *block = nullptr;
    rc = static_scratch_address(&block);
    if (rc != GD_OK) return rc;
    const gd_map_desc &m = r->dm.d;
    const bool decals = lanes->decal_slots > 0 && lanes->decal_state && lanes->decal_geom && r->overlays.d.decal_variant_count > 0;
    Scratch sc = r->sc;   // keeps the renderer's status word
    const bool fused = r->assembly == GD_ASSEMBLY_FUSED;
    auto carve = [&](unsigned char *at, size_t L) { return carve_scratch(sc, at, L, m, r->dm.masked_count, decals, fused, STATIC_SPILL_BLOCKS); };
    const size_t one = carve(nullptr, 1), two = carve(nullptr, 2);
    if (one > STATIC_SCRATCH_BYTES)
        return fail(GD_E_ARG, "map too large for gd_render_static: one lane needs " + std::to_string(one) + " bytes of working memory, the static block holds " +
                                  std::to_string(STATIC_SCRATCH_BYTES));
    // the layout grows by a fixed amount per lane, up to the padding between its buffers
    size_t fit = 1 + (STATIC_SCRATCH_BYTES - one) / (two - one);
    while (fit > 1 && carve(nullptr, fit) > STATIC_SCRATCH_BYTES) --fit;
    const int chunk = fit > 4096 ? 4096 : (int)fit;
    if (lanes->lane_count > GD_STATIC_MAX_LANES)
        return fail(GD_E_ARG, "gd_render_static renders at most " + std::to_string(GD_STATIC_MAX_LANES) + " lanes per call");
    carve(block, (size_t)chunk);
    hipStream_t caller = static_cast<hipStream_t>(stream);
    // the block keeps whatever the last call left: the kernels expect nothing of it
    for (int base = 0; base < lanes->lane_count; base += chunk) {
        const int count = lanes->lane_count - base < chunk ? lanes->lane_count - base : chunk;
        rc = launch_chunk(r, sc, lanes, out, base, count, caller, false);
        if (rc != GD_OK) return rc;
    }
    return GD_OK;
}

int gd_render_timed(gd_renderer *r, const gd_lanes_desc *lanes, const gd_frame_out *out, void *stream, int32_t launches, float *ms, int32_t stage_count) {
    int rc = check_render_args(r, lanes, out);
    if (rc != GD_OK) return rc;
    if (r->chunk_lanes <= 0) return fail(GD_E_ARG, "this renderer was created for 0 lanes and holds no working memory");
    if (!ms || stage_count < STAGE_COUNT - 1 || launches <= 0) return fail(GD_E_ARG, "ms must hold 8 stage times");
    for (int s = 0; s < stage_count; ++s) ms[s] = 0.0f;
    hipStream_t st = static_cast<hipStream_t>(stream);
    for (int it = 0; it < launches; ++it) {
        for (int base = 0; base < lanes->lane_count; base += r->chunk_lanes) {
            int count = lanes->lane_count - base < r->chunk_lanes ? lanes->lane_count - base : r->chunk_lanes;
            rc = launch_chunk(r, r->sc, lanes, out, base, count, st, true);
            if (rc != GD_OK) return rc;
            HIP_TRY(hipEventSynchronize(r->events[STAGE_COUNT - 1]));
            for (int s = 0; s + 1 < STAGE_COUNT; ++s) {
                float t = 0.0f;
                HIP_TRY(hipEventElapsedTime(&t, r->events[s], r->events[s + 1]));
                ms[s] += t;
            }
        }
    }
    for (int s = 0; s + 1 < STAGE_COUNT; ++s) ms[s] /= (float)launches;
    return GD_OK;
}

/* Sticky status bits of the renderer: bit0 = a column had more than CAND_MAX candidate linedefs and its list was truncated.
   Replaces nothing in the reference. */
int gd_renderer_status_seen(gd_renderer *r, int32_t *status) {
    if (!r || !status) return fail(GD_E_ARG, "null argument");
    *status = (r->sc.status[STATUS_CAND_OVERFLOW] ? 1 : 0) | (r->sc.status[STATUS_PASS_OVERFLOW] ? 2 : 0);
    return GD_OK;
}

int gd_renderer_mark_status(gd_renderer *r) {
    if (!r) return fail(GD_E_ARG, "null argument");
    r->status_wanted = true;
    return GD_OK;
}

int gd_renderer_wait_status(gd_renderer *r, void *stream) {
    if (!r) return fail(GD_E_ARG, "null argument");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (r->status_marked && r->status_stream == st) HIP_TRY(hipEventSynchronize(r->status_event));
    else HIP_TRY(hipStreamSynchronize(st));
    return GD_OK;
}

/* The same once the renderer's device, which need not be the current one, has done all it was given. */
int gd_renderer_status(gd_renderer *r, int32_t *status) {
    if (!r || !status) return fail(GD_E_ARG, "null argument");
    OnDevice on(r->device);
    HIP_TRY(on.error);
    HIP_TRY(hipDeviceSynchronize());
    return gd_renderer_status_seen(r, status);
}

/* Fill the renderer's working memory with one byte value.
   Frames must not depend on what that memory held; this lets a caller check it.  Replaces nothing in the reference. */
int gd_renderer_scribble(gd_renderer *r, int32_t value, void *stream) {
    if (!r) return fail(GD_E_ARG, "null argument");
    if (!r->scratch_block) return GD_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const unsigned int byte = (unsigned int)value & 0xFFu, word = byte * 0x01010101u;
    hipLaunchKernelGGL(fill_words_kernel, dim3(4096), dim3(256), 0, st, reinterpret_cast<unsigned int *>(r->scratch_block), r->scratch_bytes / 4, word);
    if (r->sc.masked_texel)
        hipLaunchKernelGGL(fill_words_kernel, dim3(4096), dim3(256), 0, st, reinterpret_cast<unsigned int *>(r->sc.masked_texel), (size_t)r->chunk_lanes * VH * SW / 4, word);
    HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_renderer_set_assembly(gd_renderer *r, int32_t assembly) {
    if (!r) return fail(GD_E_ARG, "null argument");
    if (assembly != GD_ASSEMBLY_AUTO && assembly != GD_ASSEMBLY_FUSED && assembly != GD_ASSEMBLY_SEPARATE) return fail(GD_E_ARG, "unknown assembly");
    if (assembly == GD_ASSEMBLY_FUSED && r->chunk_lanes > 0 && r->dm.masked_count > 0 && !r->sc.masked_texel) {
        // the one plane that only this assembly uses: 65 KB a lane
        OnDevice on(r->device);
        HIP_TRY(on.error);
        if (int rc = scratch_alloc(r, (size_t)r->chunk_lanes * VH * SW, &r->sc.masked_texel)) return rc;
    }
    r->assembly = assembly;
    return GD_OK;
}

int gd_renderer_set_overlays(gd_renderer *r, const gd_overlay_desc *h) {
    if (!r || !h) return fail(GD_E_ARG, "null argument");
    SIZE_CHECK(h, gd_overlay_desc);
    if (h->weapon_patch_count < 0 || h->hud_patch_count < 0 || h->weapon_max_h < 0 || h->weapon_max_w < 0 || h->hud_max_h < 0 || h->hud_max_w < 0)
        return fail(GD_E_ARG, "negative overlay size");
    if (h->weapon_patch_count > 0 && (!h->weapon_atlas || !h->weapon_opaque || !h->weapon_w || !h->weapon_h || !h->weapon_left || !h->weapon_top))
        return fail(GD_E_ARG, "missing weapon patch array");
    if (h->decal_variant_count != 0 &&
        (h->decal_variant_count != 5 || h->decal_max_h <= 0 || h->decal_max_w <= 0 || h->decal_black_rows <= 0 || !h->decal_atlas ||
         !h->decal_h || !h->decal_left || !h->decal_top || !h->decal_opacity_lut || !h->decal_black_lut))
        return fail(GD_E_ARG, "decal patches need 5 variants, their sizes and both tables");
    if (h->decal_variant_count == 5) {
        for (int v = 0; v < 5; ++v)
            if (h->decal_h[v] < 0 || h->decal_h[v] > h->decal_max_h) return fail(GD_E_ARG, "decal height outside the atlas");
        for (int k = 0; k < 32 * 256; ++k)
            if (h->decal_opacity_lut[k] >= h->decal_black_rows) return fail(GD_E_ARG, "decal_opacity_lut names a row outside decal_black_lut");
    }
    if (h->hud_patch_count > 0 && (!h->hud_atlas || !h->hud_opaque || !h->hud_w || !h->hud_h || !h->hud_left || !h->hud_top))
        return fail(GD_E_ARG, "missing status bar patch array");
    HIP_TRY(hipDeviceSynchronize());              // no frame may still be reading the old patches
    for (void *ptr : r->overlay_allocations) (void)hipFree(ptr);
    r->overlay_allocations.clear();
    std::memset(&r->overlays, 0, sizeof(r->overlays));
    gd_overlay_desc d = *h;
    auto copy = [&](const void *host, size_t bytes, const void **device) -> int {
        void *ptr = nullptr;
        HIP_TRY(hipMalloc(&ptr, bytes ? bytes : 1));
        r->overlay_allocations.push_back(ptr);
        if (bytes) HIP_TRY(hipMemcpy(ptr, host, bytes, hipMemcpyHostToDevice));
        *device = ptr;
        return GD_OK;
    };
    int rc = GD_OK;
    const size_t wp = h->weapon_patch_count, wt = wp * h->weapon_max_h * h->weapon_max_w;
    const size_t hp = h->hud_patch_count, ht = hp * h->hud_max_h * h->hud_max_w;
#define OV(field, bytes) if (rc == GD_OK) rc = copy(h->field, (bytes), reinterpret_cast<const void **>(&d.field))
    OV(weapon_atlas, wt); OV(weapon_opaque, wt); OV(weapon_w, wp * 4); OV(weapon_h, wp * 4); OV(weapon_left, wp * 4); OV(weapon_top, wp * 4);
    OV(hud_atlas, ht); OV(hud_opaque, ht); OV(hud_w, hp * 4); OV(hud_h, hp * 4); OV(hud_left, hp * 4); OV(hud_top, hp * 4);
    r->sc.scene_depth = nullptr;
    if (h->decal_variant_count == 5) {
        OV(decal_atlas, (size_t)5 * h->decal_max_h * h->decal_max_w); OV(decal_h, 5 * 4); OV(decal_left, 5 * 4); OV(decal_top, 5 * 4);
        OV(decal_opacity_lut, 32 * 256); OV(decal_black_lut, (size_t)h->decal_black_rows * 256);
        if (rc == GD_OK) {   // the depth buffer decals test against, for one chunk of lanes
            void *ptr = nullptr;
            if (hipMalloc(&ptr, (size_t)(r->chunk_lanes > 0 ? r->chunk_lanes : 1) * VH * SW * sizeof(float)) != hipSuccess) rc = fail(GD_E_HIP, "out of device memory for the decal depth buffer");
            else { r->overlay_allocations.push_back(ptr); r->sc.scene_depth = static_cast<float *>(ptr); }
        }
    }
#undef OV
    if (rc != GD_OK) {
        for (void *ptr : r->overlay_allocations) (void)hipFree(ptr);
        r->overlay_allocations.clear();
        r->sc.scene_depth = nullptr;
        return rc;
    }
    r->overlays.d = d;
    return GD_OK;
}

int gd_renderer_set_sector_lights(gd_renderer *r, const float *lights, void *stream) {
    if (!r || !lights) return fail(GD_E_ARG, "null argument");
    HIP_TRY(hipMemcpyAsync(const_cast<float *>(r->dm.d.sector_lights), lights, (size_t)r->dm.d.sector_count * sizeof(float),
                           hipMemcpyDeviceToDevice, static_cast<hipStream_t>(stream)));
    return GD_OK;
}


int gd_observe(const uint8_t *indexed, int32_t source_rows, const uint8_t *playpal, int32_t lane_count,
               uint8_t *obs, uint8_t *frames, const uint8_t *reset_mask, int32_t stack_mode, void *stream) {
    if (stack_mode != GD_STACK_STEP && stack_mode != GD_STACK_RESET) return fail(GD_E_ARG, "unknown stack_mode");
    if (source_rows != 208 && source_rows != 240) return fail(GD_E_ARG, "indexed must have 208 or 240 rows");
    if (lane_count < 0) return fail(GD_E_ARG, "negative lane count");
    if (lane_count == 0) return GD_OK;    // an empty batch: its tensors may have no address
    if (!indexed || !playpal) return fail(GD_E_ARG, "null argument");
    if (!obs && !frames) return GD_OK;
    for (int base = 0; base < lane_count; base += 32768) {
        int count = lane_count - base < 32768 ? lane_count - base : 32768;
        const size_t F = (size_t)GD_OBS_SIZE * GD_OBS_SIZE;
        launch_observe(static_cast<hipStream_t>(stream), indexed + (size_t)base * source_rows * SW, (size_t)source_rows * SW, source_rows, playpal, count,
                       obs ? obs + (size_t)base * F : nullptr, frames ? frames + (size_t)base * GD_FRAME_STACK * F : nullptr,
                       reset_mask ? reset_mask + base : nullptr, stack_mode, nullptr, false, nullptr);
    }
    HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_expand_rgb24(const uint8_t *indexed, int32_t rows, const uint8_t *playpal, int32_t lane_count, uint8_t *rgb, void *stream) {
    if (rows <= 0 || lane_count < 0) return fail(GD_E_ARG, "bad shape");
    size_t pixels = (size_t)lane_count * rows * SW;
    if (pixels == 0) return GD_OK;        // an empty batch: its tensors may have no address
    if (!indexed || !playpal || !rgb) return fail(GD_E_ARG, "null argument");
    const size_t step = (size_t)320 << 22;   // whole rows
    for (size_t base = 0; base < pixels; base += step) {
        size_t count = pixels - base < step ? pixels - base : step;
        hipLaunchKernelGGL(expand_rgb_kernel, dim3((unsigned)((count + EXPAND_PIXELS - 1) / EXPAND_PIXELS)), dim3(EXPAND_THREADS), 0, static_cast<hipStream_t>(stream),
                           indexed + base, playpal, count, rgb + base * 3, nullptr, (size_t)1);
    }
    HIP_TRY(hipGetLastError());
    return GD_OK;
}

namespace {
int pack_actors(const gd_actor_desc *a, const gd_facing_desc *facing, void *stream) {
    const int32_t counts[] = {a->lane_count, a->enemy_slots, a->doll_count, a->player_projectile_slots, a->enemy_projectile_slots,
                              a->fog_slots, a->puff_slots, a->item_count, a->drop_slots};
    for (int32_t v : counts) if (v < 0) return fail(GD_E_ARG, "negative count");
    if (a->attack_frames < 3 || a->death_frames < 1 || a->xdeath_frames < 1 || a->explosion_frames < 1)
        return fail(GD_E_ARG, "animation tables need at least 3 attack frames and 1 frame of every other kind");
    // every pointer of the descriptor sits between the scalars and the end of the struct
    const auto at = [](const void *field) { return static_cast<const void *const *>(field); };
    for (const void *const *p = at(&a->enemy_x); p <= at(&a->sprite_style); ++p) {
        const bool doll = p >= at(&a->doll_x) && p <= at(&a->doll_rotation);
        const bool item = p >= at(&a->item_x) && p <= at(&a->item_animation_initial_tics);
        const bool rotation = p == at(&a->enemy_rotation) || p == at(&a->doll_rotation) || p == at(&a->projectile_rotation) || p == at(&a->enemy_projectile_rotation);
        if (!*p && !(doll && a->doll_count == 0) && !(item && a->item_count == 0) && !(rotation && facing)) return fail(GD_E_ARG, "null tensor in gd_actor_desc");
    }
    if (facing) {
        if (facing->doll_stride < 0 || facing->item_stride < 0) return fail(GD_E_ARG, "negative stride");
        const bool missing = !facing->x || !facing->y || !facing->enemy_angle || (!facing->doll_degrees && a->doll_count) || !facing->projectile_velocity_x ||
                             !facing->projectile_velocity_y || !facing->enemy_projectile_velocity_x || !facing->enemy_projectile_velocity_y;
        if (missing) return fail(GD_E_ARG, "null tensor in gd_facing_desc");
    }
    const long long width = 2LL * a->enemy_slots + a->doll_count + 2LL * a->player_projectile_slots + 2LL * a->enemy_projectile_slots +
                            a->fog_slots + a->puff_slots + a->item_count + a->drop_slots;
    if (a->lane_count == 0 || width == 0) return GD_OK;
    if (width > 65535 * 64LL || a->lane_count > 65535) return fail(GD_E_ARG, "too many slots or lanes for one launch");
    hipLaunchKernelGGL(facing ? pack_actors_kernel<true> : pack_actors_kernel<false>, dim3((unsigned)((width + 63) / 64), (unsigned)a->lane_count), dim3(64), 0,
                       static_cast<hipStream_t>(stream), *a, facing ? *facing : gd_facing_desc{}, (int)width);
    HIP_TRY(hipGetLastError());
    return GD_OK;
}

int pack_weapon(const gd_weapon_desc *w, unsigned narrow, void *stream) {
    if (w->lane_count < 0 || w->cooldown_slots <= 0) return fail(GD_E_ARG, "gd_weapon_desc holds a count out of range");
    const void *const needed[] = {w->active_weapon, w->weapon_state_cooldown, w->weapon_fire_count, w->weapon_ready_tics, w->weapon_lower_cooldown,
                                  w->weapon_raise_cooldown, w->pending_weapon, w->episode_time, w->player_bob_fixed, w->player_dead,
                                  w->weapon_frame_ids, w->weapon_flash_ids, w->fine_sine, w->weapon_state};
    for (const void *p : needed) if (!p) return fail(GD_E_ARG, "null tensor in gd_weapon_desc");
    if (w->flash_light && !w->weapon_flash_lights) return fail(GD_E_ARG, "flash_light needs weapon_flash_lights");
    if (w->lane_count == 0) return GD_OK;
    hipLaunchKernelGGL(pack_weapon_kernel, dim3((unsigned)((w->lane_count + 63) / 64)), dim3(64), 0, static_cast<hipStream_t>(stream), *w, narrow);
    HIP_TRY(hipGetLastError());
    return GD_OK;
}
}  // namespace

int gd_pack_actors(const gd_actor_desc *a, void *stream) {
    if (!a) return fail(GD_E_ARG, "null argument");
    SIZE_CHECK(a, gd_actor_desc);
    return pack_actors(a, nullptr, stream);
}

int gd_pack_actors_facing(const gd_actor_desc *a, const gd_facing_desc *facing, void *stream) {
    if (!a || !facing) return fail(GD_E_ARG, "null argument");
    SIZE_CHECK(a, gd_actor_desc);
    SIZE_CHECK(facing, gd_facing_desc);
    return pack_actors(a, facing, stream);
}

int gd_ray_tables(const float *angle, const float *ray_offsets, int32_t lane_count, float *ray_cos, float *ray_sin, void *stream) {
    if (lane_count < 0) return fail(GD_E_ARG, "negative lane count");
    if (lane_count == 0) return GD_OK;    // an empty batch: its tensors may have no address
    if (!angle || !ray_offsets || !ray_cos || !ray_sin) return fail(GD_E_ARG, "null argument");
    if (lane_count > INT32_MAX / SW - 1) return fail(GD_E_ARG, "too many lanes for one launch");
    const int total = lane_count * SW;
    hipLaunchKernelGGL(ray_tables_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), angle, ray_offsets, total, ray_cos, ray_sin);
    HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_sprite_depth(const float *x, const float *y, const float *angle, const float *sprite_x, const float *sprite_y,
                    int32_t lane_count, int32_t sprite_slots, float *depth, void *stream) {
    if (lane_count < 0 || sprite_slots < 0) return fail(GD_E_ARG, "negative count");
    const long long total = (long long)lane_count * sprite_slots;
    if (total == 0) return GD_OK;         // an empty batch: its tensors may have no address
    if (!x || !y || !angle || !sprite_x || !sprite_y || !depth) return fail(GD_E_ARG, "null argument");
    if (total > 256LL * INT32_MAX) return fail(GD_E_ARG, "too many billboards for one launch");
    hipLaunchKernelGGL(sprite_depth_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), x, y, angle, sprite_x, sprite_y, total,
                       sprite_slots, depth);
    HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_lane_floats(const float *x, const float *y, const float *angle, const float *ray_offsets, const float *sprite_x, const float *sprite_y, int32_t lane_count,
                   int32_t sprite_slots, float *ray_cos, float *ray_sin, float *depth, void *stream) {
    if (lane_count < 0 || sprite_slots < 0) return fail(GD_E_ARG, "negative count");
    if (lane_count == 0) return GD_OK;    // an empty batch: its tensors may have no address
    if (!angle || !ray_offsets || !ray_cos || !ray_sin) return fail(GD_E_ARG, "null argument");
    if (lane_count > INT32_MAX / SW - 1) return fail(GD_E_ARG, "too many lanes for one launch");
    const long long billboards = (long long)lane_count * sprite_slots;
    if (billboards > 0 && (!x || !y || !sprite_x || !sprite_y || !depth)) return fail(GD_E_ARG, "null argument");
    const int rays = lane_count * SW;
    const long long blocks = ((long long)rays + 255) / 256 + (billboards + 255) / 256;
    if (blocks > INT32_MAX) return fail(GD_E_ARG, "too many billboards for one launch");
    hipLaunchKernelGGL(lane_floats_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream), x, y, angle, ray_offsets, rays, ray_cos, ray_sin, sprite_x,
                       sprite_y, billboards, sprite_slots, depth);
    HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_pack_weapon(const gd_weapon_desc *w, void *stream) {
    if (!w) return fail(GD_E_ARG, "null argument");
    SIZE_CHECK(w, gd_weapon_desc);
    return pack_weapon(w, 0u, stream);
}

int gd_pack_weapon_narrow(const gd_weapon_desc *w, uint32_t narrow, void *stream) {
    if (!w) return fail(GD_E_ARG, "null argument");
    SIZE_CHECK(w, gd_weapon_desc);
    if (narrow >> 9) return fail(GD_E_ARG, "gd_weapon_desc has nine words a lane");
    return pack_weapon(w, narrow, stream);
}

int gd_pack_hud(const gd_hud_desc *h, void *stream) {
    if (!h) return fail(GD_E_ARG, "null argument");
    SIZE_CHECK(h, gd_hud_desc);
    if (h->lane_count < 0 || h->weapon_columns < 6 || h->ammo_columns < 4 || h->narrow >> 5) return fail(GD_E_ARG, "gd_hud_desc holds a count out of range");
    if (h->lane_count == 0) return GD_OK;
    const auto at = [](const void *field) { return static_cast<const void *const *>(field); };
    for (const void *const *p = at(&h->ammo_slot); p <= at(&h->hud_state); ++p) if (!*p) return fail(GD_E_ARG, "null tensor in gd_hud_desc");
    hipLaunchKernelGGL(pack_hud_kernel, dim3((unsigned)((h->lane_count + 63) / 64)), dim3(64), 0, static_cast<hipStream_t>(stream), *h);
    HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_pack_decals(const int64_t *serial, const int64_t *wall, const float *along, const float *impact_z, const int64_t *style, const float *walls,
                   int32_t wall_count, const int64_t *fine_sine, int32_t lane_count, int32_t slots, int32_t *decal_state, float *decal_geom, void *stream) {
    if (lane_count < 0 || slots < 0 || slots > (1 << 20)) return fail(GD_E_ARG, "count out of range");
    if (lane_count == 0 || slots == 0) return GD_OK;      // nothing to pack: the tensors may have no address
    if (!serial || !wall || !along || !impact_z || !style || !walls || !fine_sine || !decal_state || !decal_geom) return fail(GD_E_ARG, "null argument");
    if (wall_count <= 0) return fail(GD_E_ARG, "decals need linedefs");
    if (reinterpret_cast<uintptr_t>(walls) & 15) return fail(GD_E_ARG, "walls must lie on 16 bytes");
    hipLaunchKernelGGL(pack_decals_kernel, dim3((unsigned)lane_count), dim3(64), 0, static_cast<hipStream_t>(stream), serial, wall, along, impact_z, style, walls, wall_count,
                       fine_sine, slots, decal_state, decal_geom);
    HIP_TRY(hipGetLastError());
    return GD_OK;
}

int gd_screen_blend(const int64_t *bonus_count, const int64_t *damage_count, const float *damage_to_alpha, int32_t lane_count, float *screen_blend, void *stream) {
    if (lane_count < 0) return fail(GD_E_ARG, "negative count");
    if (lane_count == 0) return GD_OK;
    if (!bonus_count || !damage_count || !damage_to_alpha || !screen_blend) return fail(GD_E_ARG, "null argument");
    hipLaunchKernelGGL(screen_blend_kernel, dim3((unsigned)((lane_count + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), bonus_count, damage_count, damage_to_alpha,
                       lane_count, screen_blend);
    HIP_TRY(hipGetLastError());
    return GD_OK;
}

}  // extern "C"
