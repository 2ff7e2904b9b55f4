// The dipole N-body of a block of placements: dA/dt of every placement's coil at every node.
#pragma once
#include "kernels.hpp"

namespace cn {

constexpr int kClusters = 64;       // a coil's dipoles in runs of nearly equal length, one bit each
constexpr int kTopLevel = 2;        // coarsest box level: 4 x 4 x 4 boxes over the nodes' bounding box
constexpr int kMaxBoxLevels = 4;    // levels kTopLevel .. kTopLevel + 3
constexpr int kUpperOrder = 8;      // Chebyshev points per axis of the boxes above the leaves
constexpr int kLeafOrder = 6;       // ... and of the leaf boxes

// Boxes of the nodes' Morton order (a box at level l is one l-level octant, so its nodes are one
// contiguous run), from kTopLevel to the leaf level; levels = 0 where the mesh is too small for them.
struct BoxTree {
    int levels = 0;
    std::int64_t n = 0;  // nodes
    int n_box[kMaxBoxLevels] = {};
    int first[kMaxBoxLevels] = {};       // position of a level's boxes in the arrays below
    int total = 0;
    double half[kMaxBoxLevels][3] = {};  // half widths (mm)
    DeviceBuffer<double> center;         // (total, 3) mm
    DeviceBuffer<std::int32_t> parent;   // -1 at the top
    DeviceBuffer<std::int32_t> octant;   // position in the parent: bit a set = upper half along axis a
    DeviceBuffer<double> rule;           // admissibility distance of a level's boxes (m), per level
    DeviceBuffer<float> tables;          // Chebyshev points and parent-to-child interpolation (see dipole.hip)
    int n_chunks = 0;                    // 64-node pieces of the leaves
    DeviceBuffer<std::int32_t> chunk_node, chunk_end, chunk_leaf;
    DeviceBuffer<double> chunk_ball;     // (n_chunks, 4) bounding balls (mm)
};

void build_box_tree(BoxTree& t, const double* nodes_mm, std::int64_t n, hipStream_t s);

// One coil on the device in its own frame, and the buffers of a block's N-body.
struct DipoleSet {
    int n = 0;
    bool parallel = false;  // every moment lies along `dir`
    bool boxes = false;     // clustered for the box method
    double dir[3] = {0.0, 0.0, 0.0};
    DeviceBuffer<double> coil;     // (n, 6) positions (m) and moments, in cluster order
    DeviceBuffer<double> spheres;  // (kClusters, 4) bounding spheres (m)
    DeviceBuffer<double> frames;   // (k, 16)
    DeviceBuffer<std::int32_t> order;  // the caller's index of each
    DeviceBuffer<float4> wide, close;  // a block's dipoles in world axes, for the box and the node sums
    DeviceBuffer<float4> given;        // ... and in the caller's order (moments that differ in direction)
    DeviceBuffer<double> origin;   // (k, 3) m
    DeviceBuffer<float> dirs;      // (k, 3)
    DeviceBuffer<unsigned long long> far;  // (boxes, k) clusters taken through a box or its ancestors
    DeviceBuffer<float> values[kMaxBoxLevels];
    DeviceBuffer<std::int32_t> near, near_count;  // (k, chunks) chunks summed in the caller's order; (k)
    DeviceBuffer<unsigned char> near_flag;        // (chunks, k)
    PinnedStage stage_coil, stage_frames;
};

// The coil of the following dadt_block calls: positions (m) and moments, (n_dip, 3) each, on the host.
void set_coil(DipoleSet& d, const BoxTree& t, const double* pos_m, const double* mom,
              std::int64_t n_dip, hipStream_t s);

// out (n, 3, K) = scale sum_j m_j x (r - s_j) / |r - s_j|^3 for the k placements with coil frames tf
// (k x 16, host; columns past k are zero). max_blocks > 0 caps the grid of the passes over the nodes (not
// that of the box passes before them); `beside` keeps the footprint small next to a solve on another
// stream.
void dadt_block(DipoleSet& d, const BoxTree& t, const double* nodes_mm, std::int64_t n, const double* tf, int k, int K,
                float scale, float* out, int max_blocks, bool beside, hipStream_t s);

}  // namespace cn
