// Internal types shared by the runtime translation units (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "common.hpp"
#include "transfer_blas_kernels.hpp"

namespace sfem_amd {

// ----------------------------------------------------------------- device memory helper
template <typename T>
struct DevArray {
    T *p{nullptr};
    size_t n{0};
    DevArray() = default;
    DevArray(const DevArray &) = delete;
    DevArray &operator=(const DevArray &) = delete;
    ~DevArray() { reset(); }
    void reset() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    int alloc(size_t count) {
        reset();
        if (count == 0) return SFEM_SUCCESS;
        SFEM_AMD_HIP_CHECK(hipMalloc((void **)&p, sizeof(T) * count));
        n = count;
        return SFEM_SUCCESS;
    }
    int upload(const T *h, size_t count) {
        if (alloc(count)) return SFEM_FAILURE;
        // host or device source (unified addressing)
        if (count) SFEM_AMD_HIP_CHECK(sync_memcpy(p, h, sizeof(T) * count, hipMemcpyDefault));
        return SFEM_SUCCESS;
    }
};

inline double *reduction_ws() {
    static double *ws = nullptr;
    if (!ws) {
        if (hipMalloc((void **)&ws, sizeof(double) * reduction_workspace_doubles()) != hipSuccess) ws = nullptr;
    }
    return ws;
}

inline int fill_zero(void *p, size_t bytes, hipStream_t s) {
    return blas_values<float>((ptrdiff_t)(bytes / sizeof(float)), 0.f, (float *)p, s);
}

inline uint16_t to_bf16(float f) {
    // round to nearest even
    uint32_t u;
    std::memcpy(&u, &f, 4);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);
    const uint32_t lsb = (u >> 16) & 1u;
    u += 0x7fffu + lsb;
    return (uint16_t)(u >> 16);
}

// ----------------------------------------------------------------- operator base
struct OpBase {
    virtual ~OpBase() = default;
    virtual int apply(const void *x, void *y, hipStream_t s) = 0;
    // y = A x (overwriting y).  Default: zero y, then accumulate; operators whose kernels own
    // every output entry override it and skip both the fill and the read of y.
    virtual int apply_overwrite(const void *x, void *y, hipStream_t s) {
        if (fill_zero(y, (size_t)rows() * (real_type() == SFEM_AMD_FLOAT64 ? 8 : 4), s)) return SFEM_FAILURE;
        return apply(x, y, s);
    }
    virtual ptrdiff_t rows() const = 0;
    virtual ptrdiff_t cols() const { return rows(); }
    virtual int real_type() const = 0;
    virtual int diag(void *, hipStream_t) {
        set_last_error("diag not available for this operator");
        return SFEM_FAILURE;
    }
    virtual int block_diag(void *, hipStream_t) {
        set_last_error("block diagonal not available for this operator");
        return SFEM_FAILURE;
    }
    // sshex8 operators: the mesh whose skeleton gather writes their shared nodes (Dirichlet rows on
    // it can be set there, see apply_constrained); null otherwise
    virtual const sfem_amd_mesh *gather_mesh(hipStream_t) { return nullptr; }
    virtual int block_size() const { return 1; }
    // operators whose overwriting apply writes every node in one pass: Dirichlet rows as a byte per mesh node
    // (bit per component) in apply_constrained (overwriting only), in place of gather_mesh's skeleton entries
    virtual bool masks_nodes(hipStream_t) { return false; }
    // y (+)= A x with the rows flagged in cmask (per entry of gather_mesh's skeleton or, with masks_nodes,
    // per node; bit per component) set to x instead; overwrite: y is output only
    virtual int apply_constrained(const void *, void *, const uint8_t *, int, hipStream_t) {
        set_last_error("constrained gather not available for this operator");
        return SFEM_FAILURE;
    }
    // Prolongations: y += P x with constrained fine rows unchanged (the multigrid's coarse
    // correction in one pass), where adds_correction says so.
    virtual bool adds_correction(hipStream_t) { return false; }
    virtual int apply_add(const void *, void *, hipStream_t) {
        set_last_error("adding prolongation not available for this operator");
        return SFEM_FAILURE;
    }
    // A Chebyshev3 step run inside the apply (ChebStep: with t = A x, p and x updated in place, t
    // not stored); cmask as in apply_constrained.  Only where cheb3_fusable says so.
    virtual bool cheb3_fusable(hipStream_t) { return false; }
    virtual int cheb3_step(void *, const void *, const void *, void *, double, double, int, const uint8_t *,
                           hipStream_t) {
        set_last_error("fused Chebyshev step not available for this operator");
        return SFEM_FAILURE;
    }
    // Solvers and smoothers: the output holds zeros on entry to the next applies (work that
    // multiplies the initial guess may be skipped).  Other operators ignore it.
    virtual void set_initial_guess_zero(bool) {}
    // with set_initial_guess_zero(true) the output's contents are not read
    virtual bool zero_guess_ignores_x() const { return false; }
    virtual int iterations() const { return -1; }
    virtual int last_status() const { return SFEM_SUCCESS; }
    virtual const std::vector<double> *history() const { return nullptr; }
};

}  // namespace sfem_amd

namespace sfem_amd {
struct SkeletonStore {
    DevArray<int32_t> node, off, pos, ent;
    ptrdiff_t n{0};
    bool covers{false};  // every mesh node lies in some element (overwriting applies allowed)
};

// The elements of a tet4/hex8 mesh grouped into patches of neighbouring elements (patches.hip).  A patch
// kernel gathers the patch's nodes once into LDS, accumulates its elements there and adds them to y.  A slot
// is a position in the patch order of the elements.
struct ElementPatches {
    ptrdiff_t npatch{0};
    int maxloc{0};                   // largest node count of a patch
    DevArray<int32_t> start;         // [npatch + 1] slots of each patch
    DevArray<int32_t> perm;          // [E] element in each slot
    DevArray<uint16_t> lconn;        // [nv / 4][E][4] local node of each slot's corners
    DevArray<int32_t> node_off;      // [npatch + 1] ranges of the patch node lists
    DevArray<int32_t> nodes;         // mesh node of each patch node, ascending in a patch
};
// The corners of a mesh by node: node g has corners ent[off[g]] .. ent[off[g + 1] - 1], a corner being
// element * nv + local node, elements ascending.
struct NodeElements {
    DevArray<int32_t> off, ent;
};

// Making the lists above allocates and synchronises: not while the stream is being captured.
bool may_build_patches(hipStream_t s);
// Something a mesh or an operator makes at its first use, once, whichever of several threads comes first.  Once
// made it costs an apply one atomic load: no lock is taken, and what another operator or mesh is making is not
// waited for.  While the stream is being captured nothing is made and no lock is taken either.
struct LazyPart {
    // make(): 1 in use; -1 not applicable; 0 failed this time (memory, or another thread's capture), to be tried
    // again by the next call, and from the second failure on after 16, 32, ... calls
    template <typename Make>
    bool ready(hipStream_t s, Make make) {
        return ready(s, make, [] { return true; });
    }
    // due(): false to leave the making to a later call
    template <typename Make, typename Due>
    bool ready(hipStream_t s, Make make, Due due) {
        int st = state.load(std::memory_order_acquire);
        if (st) return st > 0;
        if (!due() || !may_build_patches(s)) return false;
        std::lock_guard<std::mutex> lock(making);
        st = state.load(std::memory_order_relaxed);
        if (st) return st > 0;
        if (skip > 0) {
            skip--;
            return false;
        }
        st = make();
        if (!st) {
            (void)hipGetLastError();  // the caller goes on without it
            if (failures < 16) failures++;
            skip = failures > 1 ? 8 << failures >> 1 : 0;
        }
        state.store(st, std::memory_order_release);
        return st > 0;
    }

private:
    std::atomic<int> state{0};
    std::mutex making;
    int failures{0}, skip{0};
};
}  // namespace sfem_amd

struct sfem_amd_op {
    std::shared_ptr<sfem_amd::OpBase> impl;
};

struct sfem_amd_mesh {
    int type{0};
    int level{1};
    ptrdiff_t E{0};
    ptrdiff_t nnodes{0};
    int nv{0};                             // nodes per element
    sfem_amd::DevArray<int32_t> idx;       // SoA [nv][E] (tet4/hex8) or element-major [E][nv] (sshex8)
    mutable sfem_amd::DevArray<uint16_t> count;  // incidence counts (lazy)
    mutable sfem_amd::DevArray<uint8_t> own;     // owner mask (lazy)
    const sfem_amd_mesh *parent{nullptr};        // set by sfem_amd_mesh_derefine
    // sshex8: per-node skeleton slot lists of the mesh viewed at level Lc (lazy, mesh_skeleton)
    mutable std::map<int, std::unique_ptr<sfem_amd::SkeletonStore>> skel;
    // sshex8: the macro elements cut into sub-blocks of level Ls (lazy, mesh_subblocks)
    mutable std::map<int, std::unique_ptr<sfem_amd_mesh>> sub;
    // tet4/hex8: element patches (lazy, mesh_patches and mesh_cells)
    mutable std::unique_ptr<sfem_amd::ElementPatches> patches, cells;
    mutable std::atomic<int> laplacian_applies{0};  // element by element, see cells_due
    // hex8: the elements around each node (lazy, mesh_node_elements)
    mutable std::unique_ptr<sfem_amd::NodeElements> around;
    mutable sfem_amd::LazyPart around_made;
    mutable std::mutex lists;  // held while patches or cells are made
};

namespace sfem_amd {
// Library options (sfem_amd_set_option): Chebyshev3 steps fused into the sshex8 matrix-core
// elasticity applies (default off: measured slower than the streaming update kernels).
extern bool g_fused_chebyshev;
// sshex8 Laplacian accumulating applies sum skeleton nodes with atomics (option "atomic_skeleton")
extern bool g_atomic_skeleton;
// sshex8 elasticity operators: 0 stencil form for FP64 at levels >= 10, element form otherwise; 1
// element form (matrix-core / node-wise kernels) everywhere; 2 stencil form wherever supported
// (option "elasticity_form")
extern int g_elasticity_form;
// tet4/hex8 applies on element patches (option "hex8_patches", default on) for meshes of at
// least kPatchMinElements elements; off: one element per lane with atomics.  Back-to-back applies, element-wise /
// patches: hex8 Laplacian 8,000 elements 6.8 / 8.2 us, 13,824 8.1 / 7.8, 32,768 15.1 / 7.9, 262,144 94 / 11;
// tet4 6,000 5.5 / 5.2 us, 16,464 5.7 / 4.4, 34,992 9.0 / 4.8, 279,936 48 / 6.5; FP64 hex8 elasticity 8,000
// 10 / 13 us, 13,824 17 / 14, 32,768 33 / 15.  The line lies above the crossing (about 12,000 elements)
// because little is gained near it: at 2^15 the patches' 1.3 (tet4) and 2.0 ms (hex8) are earned back after about 300
// and 280 applies on them, at 2^14 tetrahedra after 1,000.
extern int g_hex8_patches;
constexpr ptrdiff_t kPatchMinElements = (ptrdiff_t)1 << 15;
// elements per cell of mesh_cells: kHexCell hexahedra; tetrahedra as many as leave kTetCellsWanted cells, within
// kTetCellLeast and kTetCellMost (flat around these: 1.93M hexahedra at 384, 512, 768, 1,024 elements a cell
// within 4% of each other; 2.41M tetrahedra at 1,024 to 3,072 within 3%)
constexpr ptrdiff_t kHexCell = 512, kTetCellsWanted = 1024, kTetCellLeast = 512, kTetCellMost = 2048;
// Host-side state that a captured HIP graph depends on (library options, switch selections, CNN
// weights) changes the state epoch; graph-replaying operators re-capture when it moved.
uint64_t state_epoch();
void bump_state_epoch();
// Zeroes / sets constrained dofs; defined in runtime.cpp.
int constrained_set_value(const OpBase *constrained, int rt, double v, void *x, hipStream_t s);
int mesh_counts(const sfem_amd_mesh *m, hipStream_t s);
bool is_constrained(const OpBase *op);
// Builds (once) the skeleton slot lists of an sshex8 mesh from its connectivity.
int mesh_skeleton(const sfem_amd_mesh *m, int Lc);
// The sshex8 mesh's macro elements as (L/Ls)^3 sub-blocks of level Ls (sshex8_subblock_idx), built
// once per level and shared; null on failure.
const sfem_amd_mesh *mesh_subblocks(const sfem_amd_mesh *m, int Ls, hipStream_t s);
// Build (once) the element patches of a tet4/hex8 mesh (see patches.hip for the two kinds), as
// LazyPart's make() does.
int mesh_patches(const sfem_amd_mesh *m, hipStream_t s);
int mesh_cells(const sfem_amd_mesh *m, hipStream_t s);
// A Laplacian's applies run element by element until they have cost about what making the cells costs, so that a mesh
// with few applies pays for no cells and one with many at most twice what they cost.  Cells take 1.2, 2.9, 15.7 ms for
// 3.5e4, 2.0e5, 2.4e6 tetrahedra and 2.0, 3.5, 17.2 ms for 3.6e4, 2.0e5, 2.0e6 hexahedra: as long as 134, 82, 34 and
// 119, 43, 26 element-wise applies, near 30 + 3.4e6 / E for both.  The words in their order, which a further operator on
// the mesh makes at its first apply, take 0.02 to 0.2 ms (that apply is then 33 us in place of 23 for 3.5e4
// tetrahedra, 71 in place of 122 for 5.8e5).
constexpr double kCellsAfter = 30, kCellsAfterBy = 3.4e6;
// In an apply that will be repeated (GraphOp's eager one, before its recording; a benchmark's untimed ones) they are
// made at once.
struct ReplayedScope {
    bool before;
    ReplayedScope();
    ~ReplayedScope();
    ReplayedScope(const ReplayedScope &) = delete;
    ReplayedScope &operator=(const ReplayedScope &) = delete;
};
// The corners of a tet4/hex8 mesh by node, built by the first call outside a capture; null where they are not
// available (the element-wise kernels run then).
const NodeElements *mesh_node_elements(const sfem_amd_mesh *m, hipStream_t s);
sfem_amd_op *wrap_op(std::shared_ptr<OpBase> o);
}  // namespace sfem_amd
