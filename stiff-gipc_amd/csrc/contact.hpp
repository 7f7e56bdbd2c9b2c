// Contact-pair generation (Morton-cluster broad phase + distance-type narrow phase) and
// the barrier gradient/Hessian of every pair type.
#pragma once
#include "sgipc_internal.hpp"

namespace sgipc {

// The three primitive sets of the broad phase: 0 faces, 1 edges, 2 points
// (surface vertices).  Primitives are numbered set after set; in the sorted
// order every set is padded to whole clusters of 64 slots and to whole tops
// of 64 clusters.
struct BroadSets {
    int n[3] = {0, 0, 0};      // primitives
    int slot0[3] = {0, 0, 0};  // first slot
    int top0[3] = {0, 0, 0};   // first top
    int slots = 0, tops = 0;
    __host__ __device__ int start(int k) const { return k == 0 ? 0 : (k == 1 ? n[0] : n[0] + n[1]); }
    __host__ __device__ int total() const { return n[0] + n[1] + n[2]; }
    __host__ __device__ int set_of(int i) const { return i >= n[0] + n[1] ? 2 : (i >= n[0] ? 1 : 0); }
    __host__ __device__ int set_of_slot(int q) const { return q >= slot0[2] ? 2 : (q >= slot0[1] ? 1 : 0); }
    __host__ __device__ int slot_end(int k) const { return slot0[k] + (n[k] + 63) / 64 * 64; }
    __host__ __device__ int n_tops(int k) const { return (n[k] + 4095) / 4096; }
};

// Morton-sorted primitives with float boxes of leaves, clusters and tops
// (struct of arrays: lo xyz, hi xyz), each at least a float step outside the
// FP64 boxes.
struct BroadPhase {
    BroadSets sets;
    DevBuf<double> box;         // 6 per primitive: lo xyz, hi xyz
    DevBuf<int> sidx;           // primitive (inside its set) at sorted position start(set) + p
    DevBuf<float> leaf, l1, l2;
    // dir (optional): boxes swept to x - alpha dir
    void build(hipStream_t s, const double* x, const uint32_t* faces, int n_faces, const uint32_t* edges, int n_edges,
               const uint32_t* points, int n_points, const double* dir, double alpha);

  private:
    DevBuf<double> part_;
    DevBuf<uint32_t> keys_, skeys_;
    DevBuf<int> idx_;
    DevBuf<unsigned char> temp_;
};

// Counts of the reference's _cpNum: [0] pairs, [1] unused, [2] point-point,
// [3] point-edge, [4] point-triangle + edge-edge.
struct ContactCounts {
    int c[5] = {0, 0, 0, 0, 0};
};

// Max of a device array of values >= 1 (and the sum of a parallel int array).
class StepReducer {
  public:
    double max_inv(hipStream_t s, const double* v, const int* c, long n, long* total);

  private:
    DevBuf<double> part_;
    DevBuf<int> ipart_;
};

class ContactDetector {
  public:
    // Largest t in (0, 1] such that x - t dir keeps every candidate pair of
    // the surface apart (additive CCD with eta = 1 - slackness); candidates
    // from the boxes swept to x - alpha dir.
    double ccd_step(hipStream_t s, const double* x, const double* dir, double alpha, const uint32_t* faces, int n_faces,
                    const uint32_t* edges, int n_edges, const uint32_t* surf, int n_surf, const int* body_id,
                    const int* btype, double dhat_sq, double slackness, long* n_candidates);
    // Pairs within squared distance dhat_sq; writes at most `capacity` pairs
    // and their MatIndex.  Order: point-face pairs by (surface slot, face),
    // then edge-edge pairs by (edge, edge).  Throws SGIPC_CAPACITY (counts
    // filled) when capacity is short.
    ContactCounts detect(hipStream_t s, const double* x, const double* rest, int n_verts, const uint32_t* faces,
                         int n_faces, const uint32_t* edges, int n_edges, const uint32_t* surf, int n_surf,
                         const int* body_id, const int* btype, double dhat_sq, int* pairs, int* mat_index,
                         int capacity);
    // pair count of the last detection, also when it threw SGIPC_CAPACITY
    int last_total = 0;

  private:
    BroadPhase broad_;
    long raw_cap_ = 0;  // entries of the unsorted pair buffer
    DevBuf<int> cnt_, total_;
    DevBuf<uint64_t> rkey_, rkey_sorted_;
    DevBuf<int> rid_, rid_sorted_;
    DevBuf<int4> rpair_;
    DevBuf<uint64_t> cls_, cls_scan_;
    DevBuf<unsigned char> temp_;
    DevBuf<double> vals_;
    StepReducer red_;
};

// Ground step (largest t keeping surface vertices above normal . x = offset
// with the reference's slackness rule) and tet injectivity step.
double ground_step(hipStream_t s, StepReducer& red, DevBuf<double>& vals, const double* x, const uint32_t* surf,
                   int n_surf, const double* normal, double offset, const double* dir, double slackness);
double injective_step(hipStream_t s, StepReducer& red, DevBuf<double>& vals, const double* x, const uint32_t* tets,
                      int n_tets, const double* dir, double slackness, double error_rate);

// Barrier gradient (atomically added into grad when non-null) and the
// Hessian blocks of every pair type into the contact arena
// [PT + EE x 16 | PE x 9 | PP x 4] by MatIndex (n4, n3: PT+EE and PE counts);
// lower blocks are moved to (col, row) and zeroed.
void launch_barrier_pairs(hipStream_t s, int n_pairs, const double* x, const int* pairs, const int* mat_index, int n4,
                          int n3, double dhat_sq, double kappa, int hess_offset, double* grad, double* tvals,
                          int* trows, int* tcols, int* bad);

}  // namespace sgipc
