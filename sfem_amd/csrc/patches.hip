// Element patches of tet4/hex8 meshes: the partitions that the patch kernels of
// unstructured_kernels.hip run on.  Two of them, by what the kernel on top is bound by:
//   cells   (the Laplacians) neighbourhoods of seeds, grown on the device in a few milliseconds, of
//           any size around a mean;
//   patches (hex8 elasticity, bound by its arithmetic) full patches of 512 elements, two rounds of a
//           256-thread block, with the fewest shared nodes; grown in order on the host, tenths of a
//           second for millions of elements.
// Both end in assemble(): elements sorted by patch, patch node lists and local numbering, on the device.
// Setup only, once per mesh, deterministic.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <climits>
#include <vector>

#include "common.hpp"
#include "internal.hpp"
#include "unstructured_kernels.hpp"

namespace sfem_amd {
namespace {

#define GRID_LOOP(i, n)                                                                                 \
    for (ptrdiff_t i = (ptrdiff_t)blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += (ptrdiff_t)gridDim.x * blockDim.x)

template <typename T>
__global__ void fill_kernel(const ptrdiff_t n, const T v, T *__restrict__ a) {
    GRID_LOOP(i, n) a[i] = v;
}
__global__ void iota_kernel(const ptrdiff_t n, int32_t *__restrict__ a) {
    GRID_LOOP(i, n) a[i] = (int32_t)i;
}
struct MaxI32 {
    __host__ __device__ int32_t operator()(int32_t a, int32_t b) const { return a > b ? a : b; }
};

// hipCUB calls with a scratch buffer that grows as needed
struct Scratch {
    DevArray<unsigned char> tmp;
    template <typename F>
    int run(F f) {
        size_t need = 0;
        SFEM_AMD_HIP_CHECK(f(nullptr, need));
        if (need > tmp.n && tmp.alloc(need)) return SFEM_FAILURE;
        SFEM_AMD_HIP_CHECK(f((void *)tmp.p, need));
        return SFEM_SUCCESS;
    }
    template <typename K>
    int sort(const K *kin, K *kout, const int32_t *vin, int32_t *vout, ptrdiff_t n, int bits, hipStream_t s) {
        return run([&](void *t, size_t &b) {
            return hipcub::DeviceRadixSort::SortPairs(t, b, kin, kout, vin, vout, (int)n, 0, bits, s);
        });
    }
    int exclusive_sum(const int32_t *in, int32_t *out, ptrdiff_t n, hipStream_t s) {
        return run([&](void *t, size_t &b) { return hipcub::DeviceScan::ExclusiveSum(t, b, in, out, (int)n, s); });
    }
    int inclusive_sum(const int32_t *in, int32_t *out, ptrdiff_t n, hipStream_t s) {
        return run([&](void *t, size_t &b) { return hipcub::DeviceScan::InclusiveSum(t, b, in, out, (int)n, s); });
    }
};
int bits_for(int64_t n) {  // bits of the values 0 .. n
    int b = 1;
    while (b < 63 && (n >> b)) b++;
    return b;
}
int fetch(const int32_t *d, int32_t *h, hipStream_t s) {
    SFEM_AMD_HIP_CHECK(hipMemcpyAsync(h, d, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    SFEM_AMD_HIP_CHECK(hipStreamSynchronize(s));
    return SFEM_SUCCESS;
}
#define LAUNCH(kernel, n, ...)                                  \
    do {                                                        \
        kernel<<<grid_for(n), kBlock, 0, s>>>(n, __VA_ARGS__);  \
        SFEM_AMD_HIP_CHECK(hipGetLastError());                  \
    } while (0)

// ---------------------------------------------------------------- assembly
// run starts of the sorted labels (position of each run's first entry, else 0)
__global__ void label_runs_kernel(const ptrdiff_t n, const int32_t *__restrict__ label, int32_t *__restrict__ at) {
    GRID_LOOP(i, n) at[i] = i > 0 && label[i] != label[i - 1] ? (int32_t)i : 0;
}
// a patch starts at each run and every cap entries inside it
__global__ void patch_heads_kernel(const ptrdiff_t n, const int32_t *__restrict__ run, const int cap,
                                   int32_t *__restrict__ head) {
    GRID_LOOP(i, n) head[i] = (i - run[i]) % cap == 0;
}
__global__ void patch_starts_kernel(const ptrdiff_t n, const int32_t *__restrict__ head,
                                    const int32_t *__restrict__ incl, int32_t *__restrict__ start) {
    GRID_LOOP(i, n) {
        if (head[i]) start[incl[i] - 1] = (int32_t)i;
        if (i == n - 1) start[incl[i]] = (int32_t)n;
    }
}
// keys (patch, node) of every corner of the sorted elements
__global__ void corner_keys_kernel(const ptrdiff_t n, const ptrdiff_t E, const int nv, const int nbits,
                                   const int32_t *__restrict__ perm, const int32_t *__restrict__ incl,
                                   const int32_t *__restrict__ idx, uint64_t *__restrict__ key,
                                   int32_t *__restrict__ pos) {
    GRID_LOOP(i, n) {
        const ptrdiff_t v = i / E, slot = i - v * E;
        key[i] = ((uint64_t)(incl[slot] - 1) << nbits) | (uint32_t)idx[v * E + perm[slot]];
        pos[i] = (int32_t)i;
    }
}
__global__ void key_heads_kernel(const ptrdiff_t n, const uint64_t *__restrict__ key, int32_t *__restrict__ head) {
    GRID_LOOP(i, n) head[i] = i == 0 || key[i] != key[i - 1];
}
// patch node lists and their ranges
__global__ void node_lists_kernel(const ptrdiff_t n, const int nbits, const uint64_t *__restrict__ key,
                                  const int32_t *__restrict__ incl, int32_t *__restrict__ nodes,
                                  int32_t *__restrict__ node_off) {
    GRID_LOOP(i, n) {
        const uint64_t k = key[i];
        if (i == 0 || k != key[i - 1]) {
            const int32_t u = incl[i] - 1, g = (int32_t)(k & (((uint64_t)1 << nbits) - 1));
            nodes[u] = g;
            if (i == 0 || (k >> nbits) != (key[i - 1] >> nbits)) node_off[k >> nbits] = u;
        }
        if (i == n - 1) node_off[(k >> nbits) + 1] = incl[i];
    }
}
// local nodes, [nv / 4][E][4]
__global__ void local_nodes_kernel(const ptrdiff_t n, const ptrdiff_t E, const int nbits,
                                   const uint64_t *__restrict__ key, const int32_t *__restrict__ pos,
                                   const int32_t *__restrict__ incl, const int32_t *__restrict__ node_off,
                                   uint16_t *__restrict__ lconn) {
    GRID_LOOP(i, n) {
        const ptrdiff_t v = pos[i] / E, slot = pos[i] - v * E;
        lconn[((v / 4) * E + slot) * 4 + v % 4] = (uint16_t)(incl[i] - 1 - node_off[key[i] >> nbits]);
    }
}
__global__ void list_sizes_kernel(const ptrdiff_t n, const int32_t *__restrict__ off, int32_t *__restrict__ size) {
    GRID_LOOP(i, n) size[i] = off[i + 1] - off[i];
}

// label: element -> group (device, destroyed); groups become patches of at most cap elements.  never: it fails
// for this mesh whenever it is tried
int assemble(const sfem_amd_mesh *m, DevArray<int32_t> &label, int64_t max_label, int cap, ElementPatches &pt,
             bool &never, hipStream_t s) {
    const int nv = m->nv;
    const ptrdiff_t E = m->E, N = m->nnodes, n = E * nv;
    Scratch sc;
    DevArray<int32_t> a, b, head, incl, pos, spos;
    // elements by group, ascending ids within one (consecutive slots are consecutive elements wherever the
    // mesh allows)
    if (a.alloc(E) || b.alloc(E) || head.alloc(n) || incl.alloc(n) || pt.perm.alloc(E)) return SFEM_FAILURE;
    LAUNCH(iota_kernel, E, a.p);
    if (sc.sort(label.p, b.p, a.p, pt.perm.p, E, bits_for(max_label), s)) return SFEM_FAILURE;
    LAUNCH(label_runs_kernel, E, b.p, label.p);
    if (sc.run([&](void *t, size_t &bytes) {
            return hipcub::DeviceScan::InclusiveScan(t, bytes, label.p, a.p, MaxI32(), (int)E, s);
        }))
        return SFEM_FAILURE;
    LAUNCH(patch_heads_kernel, E, a.p, cap, head.p);
    if (sc.inclusive_sum(head.p, b.p, E, s)) return SFEM_FAILURE;
    int32_t np = 0;
    if (fetch(b.p + E - 1, &np, s)) return SFEM_FAILURE;
    pt.npatch = np;
    if (pt.start.alloc((size_t)np + 1) || pt.node_off.alloc((size_t)np + 1)) return SFEM_FAILURE;
    LAUNCH(patch_starts_kernel, E, head.p, b.p, pt.start.p);
    // patch node lists, ascending, and local numbering
    const int nbits = bits_for(N);
    DevArray<uint64_t> key, skey;
    if (key.alloc(n) || skey.alloc(n) || pos.alloc(n) || spos.alloc(n) || pt.lconn.alloc(n))
        return SFEM_FAILURE;
    LAUNCH(corner_keys_kernel, n, E, nv, nbits, pt.perm.p, b.p, m->idx.p, key.p, pos.p);
    if (sc.sort(key.p, skey.p, pos.p, spos.p, n, nbits + bits_for(np), s)) return SFEM_FAILURE;
    LAUNCH(key_heads_kernel, n, skey.p, head.p);
    if (sc.inclusive_sum(head.p, incl.p, n, s)) return SFEM_FAILURE;
    int32_t total = 0;
    if (fetch(incl.p + n - 1, &total, s)) return SFEM_FAILURE;
    if (pt.nodes.alloc(total)) return SFEM_FAILURE;
    LAUNCH(node_lists_kernel, n, nbits, skey.p, incl.p, pt.nodes.p, pt.node_off.p);
    LAUNCH(local_nodes_kernel, n, E, nbits, skey.p, spos.p, incl.p, pt.node_off.p, pt.lconn.p);
    LAUNCH(list_sizes_kernel, (ptrdiff_t)np, pt.node_off.p, head.p);
    if (sc.run([&](void *t, size_t &bytes) { return hipcub::DeviceReduce::Max(t, bytes, head.p, incl.p, (int)np, s); }))
        return SFEM_FAILURE;
    int32_t maxloc = 0;
    if (fetch(incl.p, &maxloc, s)) return SFEM_FAILURE;
    if (maxloc > 65535) {
        never = true;
        set_last_error("element patches: more than 65535 nodes in a patch");
        return SFEM_FAILURE;
    }
    pt.maxloc = maxloc;
    SFEM_AMD_HIP_CHECK(hipStreamSynchronize(s));
    return SFEM_SUCCESS;
}

// ---------------------------------------------------------------- cells
// C. Wellons' "lowbias32" integer hash (published with his search for hash functions of this form, 2018)
__host__ __device__ __forceinline__ uint32_t mix32(uint32_t h) {
    h ^= h >> 16;
    h *= 0x7feb352du;
    h ^= h >> 15;
    h *= 0x846ca68bu;
    return h ^ (h >> 16);
}
// Growth keys: (round, label in a scrambled order), so that a node keeps the labels of the first round
// that reached it and ties inside a round favour no side.  The scramble is a bijection of 20 bits.
constexpr int kLabelBits = 20;
constexpr uint32_t kLabelMask = (1u << kLabelBits) - 1, kScramble = 0x9E379u, kUnscramble = 0x16C9u;
static_assert(((uint64_t)kScramble * kUnscramble & kLabelMask) == 1, "inverse modulo 2^20");
constexpr int kMaxRounds = (1 << (32 - kLabelBits)) - 2;
constexpr uint32_t kNoKey = 0xffffffffu;
constexpr uint32_t kScramble32 = 0x9E3779B1u, kUnscramble32 = 0x0E8B2F51u;  // likewise for element ids
static_assert((uint32_t)(kScramble32 * kUnscramble32) == 1u, "inverse modulo 2^32");

__global__ void seed_flags_kernel(const ptrdiff_t E, const uint32_t below, int32_t *__restrict__ flag) {
    GRID_LOOP(e, E) flag[e] = e == 0 || mix32((uint32_t)e) < below;
}
__global__ void seed_list_kernel(const ptrdiff_t E, const int32_t *__restrict__ flag, const int32_t *__restrict__ rank,
                                 int32_t *__restrict__ seed) {
    GRID_LOOP(e, E) if (flag[e]) seed[rank[e]] = (int32_t)e;
}
__global__ void plant_kernel(const ptrdiff_t K, const int32_t *__restrict__ seed, int32_t *__restrict__ label,
                             int32_t *__restrict__ dist) {
    GRID_LOOP(k, K) {
        label[seed[k]] = (int32_t)k;
        dist[seed[k]] = 0;
    }
}
// the elements reached in round r offer their label to their nodes
__global__ void grow_nodes_kernel(const ptrdiff_t E, const int nv, const int r, const int32_t *__restrict__ idx,
                                  const int32_t *__restrict__ label, const int32_t *__restrict__ dist,
                                  uint32_t *__restrict__ nkey) {
    GRID_LOOP(e, E) {
        if (dist[e] != r) continue;
        const uint32_t k = ((uint32_t)r << kLabelBits) | (((uint32_t)label[e] * kScramble) & kLabelMask);
        for (int v = 0; v < nv; v++) {
            const int32_t g = idx[v * E + e];
            if (nkey[g] > k) atomicMin(&nkey[g], k);
        }
    }
}
// unreached elements take the least key of their nodes; left counts those that found none
__global__ void grow_elements_kernel(const ptrdiff_t E, const int nv, const int r, const int32_t *__restrict__ idx,
                                     const uint32_t *__restrict__ nkey, int32_t *__restrict__ label,
                                     int32_t *__restrict__ dist, int32_t *__restrict__ left) {
    int miss = 0;
    GRID_LOOP(e, E) {
        if (dist[e] >= 0) continue;
        uint32_t k = kNoKey;
        for (int v = 0; v < nv; v++) k = min(k, nkey[idx[v * E + e]]);
        if (k == kNoKey) {
            miss++;
            continue;
        }
        label[e] = (int32_t)((k & kLabelMask) * kUnscramble & kLabelMask);
        dist[e] = r + 1;
    }
    for (int o = 32; o > 0; o >>= 1) miss += __shfl_xor(miss, o);
    if ((threadIdx.x & 63) == 0 && miss) atomicAdd(left, miss);
}
// components without a seed: groups of consecutive elements (the element ids are all that relates them)
__global__ void label_rest_kernel(const ptrdiff_t E, const int32_t first, int32_t *__restrict__ label,
                                  int32_t *__restrict__ dist) {
    GRID_LOOP(e, E) if (dist[e] < 0) {
        label[e] = first + (int32_t)(e / kPatchElements);
        dist[e] = 0;
    }
}
// nodes between cells (depth 0) and inside one
__global__ void node_span_kernel(const ptrdiff_t E, const int nv, const int32_t *__restrict__ idx,
                                 const int32_t *__restrict__ label, int32_t *__restrict__ lo, int32_t *__restrict__ hi) {
    GRID_LOOP(e, E)
    for (int v = 0; v < nv; v++) {
        const int32_t g = idx[v * E + e];
        atomicMin(&lo[g], label[e]);
        atomicMax(&hi[g], label[e]);
    }
}
__global__ void node_depth_kernel(const ptrdiff_t N, const int32_t *__restrict__ lo, const int32_t *__restrict__ hi,
                                  uint32_t *__restrict__ nkey) {
    GRID_LOOP(g, N) nkey[g] = lo[g] < hi[g] ? 0u : kNoKey;
}
// one layer inwards from the cells' borders: elements with a node of depth r get depth r, their other
// nodes r + 1 (plain stores of one value)
__global__ void depth_kernel(const ptrdiff_t E, const int nv, const uint32_t r, const int32_t *__restrict__ idx,
                             uint32_t *__restrict__ nkey, uint32_t *__restrict__ depth, int32_t *__restrict__ changed) {
    int any = 0;
    GRID_LOOP(e, E) {
        if (depth[e] != kNoKey) continue;
        bool hit = false;
        for (int v = 0; v < nv; v++) hit |= nkey[idx[v * E + e]] == r;
        if (!hit) continue;
        depth[e] = r;
        any = 1;
        for (int v = 0; v < nv; v++) {
            const int32_t g = idx[v * E + e];
            if (nkey[g] > r + 1) nkey[g] = r + 1;
        }
    }
    if (any) *changed = 1;
}
// the deepest element of each cell (ties by a scrambled id): the next round's seed
__global__ void deepest_kernel(const ptrdiff_t E, const int32_t *__restrict__ label, const uint32_t *__restrict__ depth,
                               unsigned long long *__restrict__ best) {
    GRID_LOOP(e, E) {
        const uint32_t d = depth[e] == kNoKey ? (uint32_t)kMaxRounds : depth[e];
        const unsigned long long k = ((unsigned long long)d << 32) | ((uint32_t)e * kScramble32);
        if (best[label[e]] < k) atomicMax(&best[label[e]], k);
    }
}
__global__ void reseed_kernel(const ptrdiff_t K, const unsigned long long *__restrict__ best,
                              int32_t *__restrict__ seed) {
    GRID_LOOP(k, K) seed[k] = (int32_t)((uint32_t)best[k] * kUnscramble32);
}

}  // namespace

// Neighbourhoods of seeds: every element joins the nearest seed (breadth-first over shared nodes, all
// cells at once).  Random seeds first; then, twice, each cell's deepest element becomes its seed, which
// rounds the cells off.  Not at all, once, twice, making them and an apply: 8.1, 12.4, 17.2 ms and 48.8, 48.0,
// 47.6 us for 1.95M hexahedra; 8.1, 11.9, 15.7 ms and 32.9, 29.2, 28.8 us for 2.43M tetrahedra of a box; once and
// twice 48.0 and 46.5 us a pass for 2.41M shuffled ones.  The first time is earned back after 1,000 to 5,400 applies, the
// second after 3,000 to 12,000, and only meshes that have had many get cells at all (kCellsAfter).  hex8 box, 440
// elements a cell: 1.62, 1.58 patch nodes per element before and after (1.55 for the ordered growth of
// mesh_patches); sizes spread by a factor of about two around the mean, and cells above 2.5 times the mean are cut.
int mesh_cells(const sfem_amd_mesh *m, hipStream_t s) {
    std::lock_guard<std::mutex> lock(m->lists);
    if (m->cells) return 1;
    const ptrdiff_t E = m->E, N = m->nnodes;
    const int nv = m->nv;
    if (m->type == SFEM_AMD_SSHEX8 || E <= 0 || (double)E * nv >= 2147483647.0 || N >= 2147483647) return -1;
    // Elements per cell.  Tetrahedra, of which a hexahedron's nodes hold six: enough cells for the GPU's 256 CUs several
    // times over, and from there on larger ones, since the shared nodes' part falls with the size.
    const ptrdiff_t mean = m->type == SFEM_AMD_TET4
                                   ? std::min(std::max(E / kTetCellsWanted, kTetCellLeast), kTetCellMost)
                                   : kHexCell;
    bool never = false;
    auto build = [&]() -> std::unique_ptr<ElementPatches> {
        Scratch sc;
        DevArray<int32_t> label, dist, seed, lo, hi, counter;
        DevArray<uint32_t> nkey, depth;
        DevArray<unsigned long long> best;
        auto fail = [] { return std::unique_ptr<ElementPatches>(); };
        auto work = [&](ElementPatches &pt) -> int {
            if (label.alloc(E) || dist.alloc(E) || lo.alloc(std::max(E, N)) || hi.alloc(std::max(E, N)) ||
                nkey.alloc(N) || depth.alloc(E) || counter.alloc(1))
                return SFEM_FAILURE;
            LAUNCH(seed_flags_kernel, E, (uint32_t)(4294967295.0 / (double)mean), lo.p);
            if (sc.exclusive_sum(lo.p, hi.p, E, s)) return SFEM_FAILURE;
            int32_t last[2];
            if (fetch(hi.p + E - 1, &last[0], s) || fetch(lo.p + E - 1, &last[1], s)) return SFEM_FAILURE;
            const ptrdiff_t K = (ptrdiff_t)last[0] + last[1];
            if (K > (ptrdiff_t)kLabelMask) {
                never = true;
                set_last_error("element cells: too many cells");
                return SFEM_FAILURE;
            }
            if (seed.alloc(K) || best.alloc(K)) return SFEM_FAILURE;
            LAUNCH(seed_list_kernel, E, lo.p, hi.p, seed.p);
            int64_t max_label = K - 1;
            constexpr int kSmooth = 2;
            for (int pass = 0;; pass++) {
                LAUNCH(fill_kernel<int32_t>, E, -1, dist.p);
                LAUNCH(fill_kernel<uint32_t>, N, kNoKey, nkey.p);
                LAUNCH(plant_kernel, K, seed.p, label.p, dist.p);
                // every eighth round the host looks whether elements are left, and stops when none was reached since
                int32_t left = 0;
                int64_t before = -1;
                for (int r = 0; r < kMaxRounds; r++) {
                    LAUNCH(grow_nodes_kernel, E, nv, r, m->idx.p, label.p, dist.p, nkey.p);
                    LAUNCH(fill_kernel<int32_t>, (ptrdiff_t)1, 0, counter.p);
                    LAUNCH(grow_elements_kernel, E, nv, r, m->idx.p, nkey.p, label.p, dist.p, counter.p);
                    if (r % 8 != 7) continue;
                    if (fetch(counter.p, &left, s)) return SFEM_FAILURE;
                    if (left == 0 || left == before) break;
                    before = left;
                }
                if (left) {
                    LAUNCH(label_rest_kernel, E, (int32_t)K, label.p, dist.p);
                    max_label = K + E / kPatchElements;
                }
                // (meshes in pieces keep the first cells: the pieces without a seed have no cell to round off)
                if (pass == kSmooth || left) break;
                LAUNCH(fill_kernel<int32_t>, N, INT_MAX, lo.p);
                LAUNCH(fill_kernel<int32_t>, N, -1, hi.p);
                LAUNCH(node_span_kernel, E, nv, m->idx.p, label.p, lo.p, hi.p);
                LAUNCH(node_depth_kernel, N, lo.p, hi.p, nkey.p);
                LAUNCH(fill_kernel<uint32_t>, E, kNoKey, depth.p);
                for (int r = 0; r < kMaxRounds; r++) {
                    if (r % 4 == 0) LAUNCH(fill_kernel<int32_t>, (ptrdiff_t)1, 0, counter.p);
                    LAUNCH(depth_kernel, E, nv, (uint32_t)r, m->idx.p, nkey.p, depth.p, counter.p);
                    int32_t changed = 0;
                    if (r % 4 == 3) {
                        if (fetch(counter.p, &changed, s)) return SFEM_FAILURE;
                        if (!changed) break;
                    }
                }
                LAUNCH(fill_kernel<unsigned long long>, K, 0ull, best.p);
                LAUNCH(deepest_kernel, E, label.p, depth.p, best.p);
                LAUNCH(reseed_kernel, K, best.p, seed.p);
            }
            return assemble(m, label, max_label, (int)std::max<ptrdiff_t>(mean * 5 / 2, kPatchElements), pt, never,
                            s);
        };
        auto pt = std::make_unique<ElementPatches>();
        return work(*pt) ? fail() : std::move(pt);
    };
    m->cells = build();
    return m->cells ? 1 : never ? -1 : 0;
}

// ---------------------------------------------------------------- ordered patches
__global__ void element_major_keys_kernel(const ptrdiff_t n, const ptrdiff_t E, const int nv,
                                          const int32_t *__restrict__ idx, int32_t *__restrict__ node,
                                          int32_t *__restrict__ elem) {
    GRID_LOOP(i, n) {
        const ptrdiff_t e = i / nv;
        node[i] = idx[(i - e * nv) * E + e];
        elem[i] = (int32_t)e;
    }
}

// Breadth-first growth over shared nodes, at most kPatchElements each, the next seed taken from the
// unassigned neighbours of the previous patch (lowest id first), else the lowest unassigned element.
// On a structured box of hexahedra the patches come out as compact blocks (about 1.55 patch nodes per
// element, against 1.42 for a perfect 8^3 cube and 8 for no sharing).  A node whose elements have all
// been assigned is never looked at again, which leaves about one visit per (node, element) pair.
int mesh_patches(const sfem_amd_mesh *m, hipStream_t s) {
    std::lock_guard<std::mutex> lock(m->lists);
    if (m->patches) return 1;
    const int nv = m->nv;
    const ptrdiff_t E = m->E, N = m->nnodes, n = E * nv;
    if (m->type == SFEM_AMD_SSHEX8 || E <= 0 || (double)E * nv >= 2147483647.0 || N >= 2147483647) return -1;
    bool never = false;
    constexpr size_t P = kPatchElements;
    auto pt = std::make_unique<ElementPatches>();
    auto work = [&]() -> int {
        // node -> elements (ascending), from a sort on the device
        std::vector<int32_t> el((size_t)n), n2e((size_t)n), n2e_off((size_t)N + 1, 0), nodes((size_t)n);
        {
            Scratch sc;
            DevArray<int32_t> node, elem, snode, selem;
            if (node.alloc(n) || elem.alloc(n) || snode.alloc(n) || selem.alloc(n)) return SFEM_FAILURE;
            LAUNCH(element_major_keys_kernel, n, E, nv, m->idx.p, node.p, elem.p);
            if (sc.sort(node.p, snode.p, elem.p, selem.p, n, bits_for(N), s)) return SFEM_FAILURE;
            SFEM_AMD_HIP_CHECK(hipStreamSynchronize(s));
            SFEM_AMD_HIP_CHECK(sync_memcpy(el.data(), node.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
            SFEM_AMD_HIP_CHECK(sync_memcpy(n2e.data(), selem.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
            SFEM_AMD_HIP_CHECK(sync_memcpy(nodes.data(), snode.p, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
        }
        for (const int32_t g : nodes) n2e_off[(size_t)g + 1]++;
        for (ptrdiff_t g = 0; g < N; g++) n2e_off[g + 1] += n2e_off[g];
        std::vector<int32_t> patch_of((size_t)E, -1), queue, hint;
        std::vector<uint8_t> done((size_t)N, 0);  // every element of the node is assigned
        ptrdiff_t seed = 0;
        int32_t pid = 0;
        for (;; pid++) {
            int32_t s0 = -1;
            for (const int32_t c : hint)
                if (patch_of[c] < 0) {
                    s0 = c;
                    break;
                }
            if (s0 < 0) {
                while (seed < E && patch_of[seed] >= 0) seed++;
                if (seed >= E) break;
                s0 = (int32_t)seed;
            }
            queue.assign(1, s0);
            patch_of[s0] = pid;
            for (size_t head = 0; head < queue.size() && queue.size() < P; head++) {
                const int32_t *corner = &el[(size_t)queue[head] * nv];
                for (int v = 0; v < nv && queue.size() < P; v++) {
                    const int32_t g = corner[v];
                    if (done[g]) continue;
                    int32_t k = n2e_off[g];
                    for (; k < n2e_off[g + 1] && queue.size() < P; k++) {
                        const int32_t f = n2e[k];
                        if (patch_of[f] < 0) {
                            patch_of[f] = pid;
                            queue.push_back(f);
                        }
                    }
                    if (k == n2e_off[g + 1]) done[g] = 1;
                }
            }
            // unassigned neighbours of this patch, lowest id first
            hint.clear();
            for (const int32_t e : queue)
                for (int v = 0; v < nv; v++) {
                    const int32_t g = el[(size_t)e * nv + v];
                    if (done[g]) continue;
                    bool all = true;
                    for (int32_t k = n2e_off[g]; k < n2e_off[g + 1]; k++)
                        if (patch_of[n2e[k]] < 0) {
                            hint.push_back(n2e[k]);
                            all = false;
                        }
                    if (all) done[g] = 1;
                }
            std::sort(hint.begin(), hint.end());
            hint.erase(std::unique(hint.begin(), hint.end()), hint.end());
        }
        DevArray<int32_t> label;
        if (label.upload(patch_of.data(), patch_of.size())) return SFEM_FAILURE;
        return assemble(m, label, pid, kPatchElements, *pt, never, s);
    };
    if (work()) return never ? -1 : 0;
    m->patches = std::move(pt);
    return 1;
}

// ---------------------------------------------------------------- corners by node
__global__ void corners_kernel(const ptrdiff_t n, const ptrdiff_t E, const int nv, const int32_t *__restrict__ idx,
                               int32_t *__restrict__ node, int32_t *__restrict__ corner, int32_t *__restrict__ count) {
    GRID_LOOP(i, n) {
        const ptrdiff_t e = i / nv;
        const int32_t g = idx[(i - e * nv) * E + e];
        node[i] = g;
        corner[i] = (int32_t)i;
        atomicAdd(&count[g], 1);
    }
}
static int make_node_elements(const sfem_amd_mesh *m, hipStream_t s) {
    const ptrdiff_t E = m->E, N = m->nnodes, n = E * m->nv;
    if (m->type == SFEM_AMD_SSHEX8 || E <= 0 || (double)n >= 2147483647.0 || N >= 2147483646) return -1;
    auto ne = std::make_unique<NodeElements>();
    auto work = [&]() -> int {
        Scratch sc;
        DevArray<int32_t> node, corner, snode, count;
        if (node.alloc(n) || corner.alloc(n) || snode.alloc(n) || count.alloc(N + 1) || ne->off.alloc(N + 1) ||
            ne->ent.alloc(n))
            return SFEM_FAILURE;
        LAUNCH(fill_kernel<int32_t>, N + 1, 0, count.p);
        LAUNCH(corners_kernel, n, E, m->nv, m->idx.p, node.p, corner.p, count.p);
        if (sc.exclusive_sum(count.p, ne->off.p, N + 1, s) ||
            sc.sort(node.p, snode.p, corner.p, ne->ent.p, n, bits_for(N), s))
            return SFEM_FAILURE;
        SFEM_AMD_HIP_CHECK(hipStreamSynchronize(s));
        return SFEM_SUCCESS;
    };
    if (work()) return 0;
    m->around = std::move(ne);
    return 1;
}
const NodeElements *mesh_node_elements(const sfem_amd_mesh *m, hipStream_t s) {
    return m->around_made.ready(s, [&] { return make_node_elements(m, s); }) ? m->around.get() : nullptr;
}

bool may_build_patches(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    const hipError_t e = hipStreamIsCapturing(s, &st);
    if (e == hipErrorStreamCaptureImplicit) (void)hipGetLastError();  // a blocking stream is being captured
    return e == hipSuccess && st == hipStreamCaptureStatusNone;
}

}  // namespace sfem_amd
