// Regions: a road-like graph cut into pieces whose edges fit the registers of
// one workgroup and whose distances fit its LDS.
//
// Every vertex belongs to one region of at most kRegionVerts vertices.  The
// region's vertex list goes by falling degree, so that the 64 vertices of a
// block, which a wave handles at once, have about as many edges.  The vertices
// at positions p and p + kRegionVerts / 2, which the same thread handles, have
// adjacent local ids.  A thread of the solver holds up to kLaneEdges out-edges
// of each of its vertices.  Any further edge of a vertex is treated like an edge
// between regions, from the region to itself.
//
// A region's image, in 32-bit words:
//
//   kLaneEdges x kRegionVerts   edge k of every vertex, by position
//   kBlocks                     most edges of a block's vertices
//   nx x 3      exits: edge word of the tail, inbox slot of the edge in its
//               target region, target region
//   nin         inbox: the entered vertex, per slot
//
// Vertices are given as byte offsets (local id x 4), an edge as the offset of
// its head (exits: of its tail) | weight << kWeightShift.  An edge between two
// regions has one inbox slot, in the inbox of the region it enters; the slots
// of a region are consecutive.  Per query the solver keeps an inbox (one
// distance per slot) and one activity word per region beside the distance row.
//
// A graph is cut when the cut pays: few edges between regions (kMaxCross), every
// weight below kNoWeight, and every region within the limits below.
#pragma once

#include <stdint.h>

#include <vector>

namespace mlmq {

constexpr uint32_t kLaneEdges = 8;
constexpr uint32_t kRegionIdBits = 10;
constexpr uint32_t kRegionVerts = 1u << kRegionIdBits;
constexpr uint32_t kBlocks = kRegionVerts / 64;
constexpr uint32_t kWeightShift = 2 + kRegionIdBits;
constexpr uint32_t kOffsetMask = (1u << kWeightShift) - 4u;
constexpr uint32_t kNoWeight = ~0u >> kWeightShift;   // of an absent edge
constexpr uint32_t kRegionExits = 384;     // exits and inbox slots of a region:
constexpr uint32_t kRegionInbox = 384;     // 6 per lane of the wave that handles them
constexpr uint32_t kRegionMaxDegree = 64;
// Above this share of crossing edges the solver's messages between regions
// outweigh the relaxations kept inside them.  Road-like graphs cut at 2-5 %,
// graphs without locality at 80 % and more; nothing measured lies between.
constexpr double kMaxCross = 0.12;

struct RegionHdr {
    uint32_t first;       // first vertex in the region-ordered vertex list
    uint32_t nv, nx, nin;
    uint32_t inbox;       // first inbox slot
    uint32_t image;       // first word of the image
    uint32_t cross;       // edges to other regions
    uint32_t pad;
};

#if defined(__HIPCC__)
#define MLMQ_HD __host__ __device__
#else
#define MLMQ_HD
#endif
// Local id of position p of a region's vertex list.
MLMQ_HD inline uint32_t local_id(uint32_t p) { return p % (kRegionVerts / 2) * 2 + p / (kRegionVerts / 2); }
// Word offsets of the image's parts.
constexpr uint32_t kImageMost = kLaneEdges * kRegionVerts;
constexpr uint32_t kImageExits = kImageMost + kBlocks;
MLMQ_HD inline uint32_t image_inbox(const RegionHdr &h) { return kImageExits + 3 * h.nx; }
MLMQ_HD inline uint32_t image_words(const RegionHdr &h) { return image_inbox(h) + h.nin; }

// The cut of a graph: `order` lists the vertices region by region, region r
// holding order[first[r] .. first[r + 1]) by falling degree.
struct RegionPlan {
    std::vector<uint32_t> order;
    std::vector<uint32_t> first;
};

// Cuts a graph given by its host CSR (offsets row[0..n], destinations).
// Returns false when the graph is not worth cutting (high degrees).
bool region_plan(uint32_t n, const uint32_t *row, const uint32_t *col, RegionPlan *plan);

}  // namespace mlmq
