// Frame kernels of the particle step, written for gfx950 (wave64).
//
// One frame is four launches (five on a grid above 2^23 cells):
//   collide_kernel     one packed particle per lane, 64 consecutive ones per
//                      wavefront; `key` gives each particle's cell, so a
//                      cell is a segment of equal keys.  A cell that lies
//                      inside the wavefront is handled there: ranked by
//                      `src` (the canonical order), its first 9 particles
//                      separated (Gauss-Seidel, particles.rs:62-93), every
//                      particle finished -- integrate and limit
//                      (shaders/physics/src/particle.rs:40-82) -- and written
//                      to pos_out/vel_out at its canonical index, the new cell
//                      key computed (particles_per_cell.wgsl:14-27) and slots
//                      claimed with one atomic per neighbour direction.  A
//                      cell that runs past the wavefront's last particle is
//                      queued by size class.
//   cells_kernel       the queued cells: 65..kWideMax particles a wavefront
//                      each plus one Gauss-Seidel wavefront per three cells;
//                      2..64 particles in lane groups of 2..64 (one particle
//                      per lane); one block per larger cell.  Every path
//                      restores the canonical order (by
//                      `src`), separates the first 9 particles, finishes every
//                      particle (the overflow ones without collisions,
//                      cell.rs:79-95), writes pos_out/vel_out at the
//                      canonical index and claims slots with one atomic per
//                      neighbour direction.
//   scan_kernel        single-pass exclusive scan of the per-cell counts with
//                      decoupled look-back; writes [0, start_0.., N] and clears
//                      the counts for the next frame (prefix_sum.wgsl +
//                      cell.rs:116-131).  Large grids: cell_scan_kernel, each
//                      chunk of 1,024 cells by itself, and chunk_scan_kernel,
//                      the chunks' totals.
//   scatter_kernel     one lane per particle: dest = start[key] + slot
//                      (pack_new_particle_data.wgsl:39-44); records the source
//                      index so the next collide pass can rebuild the stable
//                      order that the reference's CPU packer defines
//                      (spatial_bin.rs:122-142), and the new cell in `key`.
//
// In-cell order.  Slots inside a new cell come from atomics, so the stored
// order is a permutation of the canonical one (ascending source index).  A
// source cell that sends several particles in one direction reserves them as
// one contiguous run with one atomic, in canonical order; the scatter flags
// the first particle of every run in bit 31 of `src`.  A cell's segment is
// therefore a handful of ascending runs whose source ranges do not
// interleave, and ordering the runs by their first source index restores the
// canonical order in O(n) (a full sort remains the fallback).
//
// Floating point: the library is compiled with -ffp-contract=off, so every
// a*b+c is a rounded multiply then a rounded add, and f32 division and
// sqrtf are the correctly rounded sequences -- the native Rust semantics of
// the reference's shader crate.
#include <hip/hip_ext.h>

#include <algorithm>
#include <atomic>

#include "frame.h"
#include "learn.h"
#include "select_nets.h"

namespace wrach {
namespace {

constexpr uint32_t kRunFlag = 0x80000000u;  // in src and in kslot.y: first of a run
constexpr uint32_t kSrcMask = 0x7fffffffu;

// ---------------------------------------------------------------------------
// Per-particle arithmetic.

// The grid of one world: its first cell key, dimensions and walls.  One
// world or a batch of equal worlds: from FrameParams; worlds of different
// sizes: from the world's WorldGrid (grid_of, below).
struct Grid {
    uint32_t base, gx, gy;
    float x1, y1;
};

// Particle::integrate + enforce_boundaries + enforce_velocity
// (shaders/physics/src/particle.rs:40-82) with the gravity/dt extension
// placed just before the integration.  A zero gravity component adds -0.0
// (FrameParams), which leaves -0.0 velocities their sign, as skipping the add
// in the reference does.  The walls are the particle's world's.
__device__ __forceinline__ void finish_particle(const FrameParams &p, const Grid &g, float &px,
                                                float &py, float &vx, float &vy) {
    vx = vx + p.gdx;
    vy = vy + p.gdy;
    px = px + vx * p.dt;
    py = py + vy * p.dt;
    if (px > g.x1) { px = g.x1; vx = vx * -1.0f; }
    if (px < p.ax) { px = p.ax; vx = vx * -1.0f; }
    if (py > g.y1) { py = g.y1; vy = vy * -1.0f; }
    if (py < p.ay) { py = p.ay; vy = vy * -1.0f; }
    if (vx < -1.0f) vx = -1.0f;
    if (vx > 1.0f) vx = 1.0f;
    if (vy < -1.0f) vy = -1.0f;
    if (vy > 1.0f) vy = 1.0f;
}


// Cell coordinates of particles_per_cell.wgsl:14-27: floor((x - ax) / cs)
// per axis, for a finished particle.  The walls leave x in [ax, x1] with
// ax = 0 and x1 = W, and the division is monotonic, so the key lies in
// [0, gx - 1] (gx - 1 = floor(W / cs) on the host, the same f32 division);
// the max only maps a NaN position, which no upload lets in, to column 0.
__device__ __forceinline__ void cell_floor(const FrameParams &p, float x, float y, float &fx, float &fy) {
    if (p.cs == 1.0f) {  // x / 1 is exact: skip the division sequence
        fx = floorf(x - p.ax);
        fy = floorf(y - p.ay);
    } else {
        fx = floorf((x - p.ax) / p.cs);
        fy = floorf((y - p.ay) / p.cs);
    }
}

__device__ __forceinline__ void cell_xy(const FrameParams &p, float x, float y, uint32_t &kx,
                                        uint32_t &ky) {
    float fx, fy;
    cell_floor(p, x, y, fx, fy);
    kx = (uint32_t)fmaxf(fx, 0.0f);
    ky = (uint32_t)fmaxf(fy, 0.0f);
}

// First cell key of the world that holds cell key c: 0 for one world; in a
// batch of equal worlds, the world's offset in the flattened key space (a
// particle never leaves its world: the walls keep it inside).
__device__ __forceinline__ uint32_t world_base(const FrameParams &p, uint32_t c) {
    if (p.world_cells == p.ncell) return 0u;
    return c / p.world_cells * p.world_cells;
}

// The grid of the world that holds cell key c (c < ncell).  Worlds of
// different sizes start on chunk boundaries, so the chunk names the world.
__device__ __forceinline__ Grid grid_of(const FrameParams &p, uint32_t c) {
    Grid g;
    if (p.grids) {
        const uint32_t last = (p.ncell - 1) >> kChunkShift;
        const uint32_t ch = (c >> kChunkShift) < last ? (c >> kChunkShift) : last;
        const WorldGrid w = p.grids[p.chunk_world[ch]];
        g.base = w.base;
        g.gx = w.gx;
        g.gy = w.gy;
        g.x1 = w.x1;
        g.y1 = w.y1;
    } else {
        g.base = world_base(p, c);
        g.gx = p.gx;
        g.gy = p.gy;
        g.x1 = p.x1;
        g.y1 = p.y1;
    }
    return g;
}

// Grid coordinates of cell key c inside its world g.
__device__ __forceinline__ void cell_coords(const Grid &g, uint32_t c, uint32_t &cx, uint32_t &cy) {
    const uint32_t l = c - g.base;
    cy = l / g.gx;
    cx = l - cy * g.gx;
}

constexpr uint32_t kNoKey = 0xffffffffu;  // no cell; cell keys stay below 2^31

// The cell of any position, kNoKey outside the grid: before a frame's step a
// loaded triple's particles may lie anywhere.
__device__ __forceinline__ uint32_t position_key(const FrameParams &p, const Grid &g, float x, float y) {
    float fx, fy;
    cell_floor(p, x, y, fx, fy);
    if (!(fx >= 0.0f && fy >= 0.0f && fx < (float)g.gx && fy < (float)g.gy)) return kNoKey;
    return g.base + (uint32_t)fy * g.gx + (uint32_t)fx;
}

// Raises a kErr* bit, for the kernels that follow and for the host, which
// looks at its words after every wait (they stay raised: the context is
// dead).  The store is visible there once the kernel has ended.
__device__ __forceinline__ void raise_error(const FrameBuffers &b, uint32_t bit) {
    atomicOr(b.error, bit);
    if (b.error_host)
        __hip_atomic_store(&b.error_host[bit == kErrLookBack ? 0 : 1], 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
}

// Claims `count` consecutive slots in cell k.  The frame's first claim in a
// chunk marks it, so that the scan visits only chunks that hold particles.
__device__ __forceinline__ uint32_t claim(const FrameBuffers &b, uint32_t k, uint32_t count) {
    const uint32_t old = atomicAdd(&b.cnt[k], count);
    if (old == 0) b.chunk_next[k >> kChunkShift] = 1;
    return old;
}

// The offset of a cell, in steps, so that a caller can have the loads of
// several cells in flight: the word that holds it (of idx, or of a large
// grid's 16-bit offsets: two cells a word), the entry in that word, on large
// grids the entry in idx where the 16 bits hold none, and the offset from
// that and the chunk's state and prefix (frame.h): an empty chunk's entries
// are stale, its cells all start at the prefix; a live chunk's are offsets,
// whole or counted from the prefix.
__device__ __forceinline__ uint32_t offset_word(const FrameBuffers &b, uint32_t k) {
    return b.off[k >> b.off_shift];
}

__device__ __forceinline__ uint32_t offset_entry(const FrameBuffers &b, uint32_t k, uint32_t word) {
    return (word >> ((k & b.off_shift) << 4)) & b.off_mask;
}

__device__ __forceinline__ uint32_t wide_entry(const FrameBuffers &b, uint32_t k, uint32_t at, uint32_t state) {
    return state == kChunkWhole || at == kWideOffset ? b.idx[k + 1] : at;
}

__device__ __forceinline__ uint32_t offset_of(uint32_t at, uint32_t state, uint32_t prefix) {
    return state == kChunkWhole ? at : state == kChunkRelative ? prefix + at : prefix;
}

// First particle of cell k (k == ncell: the end).
__device__ __forceinline__ uint32_t cell_start(const FrameParams &p, const FrameBuffers &b,
                                               uint32_t k) {
    if (k >= p.ncell) return p.n;
    const uint32_t ch = k >> kChunkShift;
    const uint32_t state = b.chunk_live[ch];
    uint32_t at = offset_entry(b, k, offset_word(b, k));
    if (b.off_shift) at = wide_entry(b, k, at, state);
    const uint32_t s = offset_of(at, state, b.chunk_prefix[ch]);
    return s < p.n ? s : p.n;
}


// Neighbour direction of a new cell relative to the old one (cx, cy) of
// world g: 0..8 for the 3x3 neighbourhood (row-major from (-1,-1)), 9 for
// anything farther.
__device__ __forceinline__ uint32_t direction(const FrameParams &p, const Grid &g, float x, float y,
                                              uint32_t cx, uint32_t cy, uint32_t &key) {
    uint32_t kx, ky;
    cell_xy(p, x, y, kx, ky);
    key = g.base + ky * g.gx + kx;
    const int dx = (int)kx - (int)cx, dy = (int)ky - (int)cy;
    if (dx < -1 || dx > 1 || dy < -1 || dy > 1) return 9;
    return (uint32_t)((dy + 1) * 3 + (dx + 1));
}

// Lane index, opaque to the optimiser: values derived from it (lane masks,
// Gauss-Seidel partners) are then recomputed where they are used instead of
// being hoisted out of the work loops and held in registers for the whole
// kernel, which spills scalar registers.
__device__ __forceinline__ uint32_t lane_id() {
    uint32_t l = threadIdx.x & 63;
    asm volatile("" : "+v"(l));
    return l;
}

__device__ __forceinline__ unsigned long long lanemask_lt() {
    return (1ull << lane_id()) - 1;
}

// Inclusive sum over the wavefront by DPP moves (lanes without a source add
// 0), one instruction a step: it stands in the latency of the scan and of the
// cell kernel's start, where six shuffles through LDS took 0.4 us a sum.
__device__ __forceinline__ uint32_t wave_inclusive_sum(uint32_t v) {
#define WRACH_DPP_ADD(ctrl, rows) \
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, rows, 0xf, false)
    WRACH_DPP_ADD(0x111, 0xf);  // row_shr:1, :2, :4, :8
    WRACH_DPP_ADD(0x112, 0xf);
    WRACH_DPP_ADD(0x114, 0xf);
    WRACH_DPP_ADD(0x118, 0xf);
    WRACH_DPP_ADD(0x142, 0xa);  // row_bcast:15 into rows 1 and 3
    WRACH_DPP_ADD(0x143, 0xc);  // row_bcast:31 into rows 2 and 3
#undef WRACH_DPP_ADD
    return v;
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Orders LDS accesses of one wavefront: its LDS instructions execute in
// program order, so a compiler fence is all a wave-private region needs.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// Cells of more than kWideMax particles: the whole block cooperates.

// Ascending bitonic sort of P (a power of two, <= kLdsSort) 64-bit keys in
// LDS.  Callers synchronise before the call; the last stage ends with a
// barrier.
__device__ void bitonic_lds(unsigned long long *sk, uint32_t P) {
    const uint32_t tid = threadIdx.x;
    for (uint32_t k = 2; k <= P; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t i = tid; i < P; i += kCollideBlock) {
                const uint32_t l = i ^ j;
                if (l > i) {
                    const unsigned long long x = sk[i], y = sk[l];
                    const bool asc = (i & k) == 0;
                    if ((x > y) == asc) {
                        sk[i] = y;
                        sk[l] = x;
                    }
                }
            }
            __syncthreads();
        }
    }
}

// Merge of two sorted runs of distinct keys into z, by the whole block (merge
// path: each thread finds its split with a binary search, then merges its
// share of the output sequentially).
__device__ void merge_block(const unsigned long long *x, uint32_t nx,
                            const unsigned long long *y, uint32_t ny,
                            unsigned long long *z) {
    const uint32_t tid = threadIdx.x;
    const uint64_t total = (uint64_t)nx + ny;
    const uint32_t d0 = (uint32_t)(total * tid / kCollideBlock);
    const uint32_t d1 = (uint32_t)(total * (tid + 1) / kCollideBlock);
    uint32_t lo = d0 > ny ? d0 - ny : 0;
    uint32_t hi = d0 < nx ? d0 : nx;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (x[mid] < y[d0 - 1 - mid]) lo = mid + 1;
        else hi = mid;
    }
    uint32_t i = lo, j = d0 - lo;
    for (uint32_t d = d0; d < d1; ++d) {
        const bool take_x = j >= ny || (i < nx && x[i] < y[j]);
        z[d] = take_x ? x[i++] : y[j++];
    }
}

// Sorts (src << 32 | local index) for a cell of n > kLdsSort particles:
// LDS-sorted chunks, then block merges ping-ponging between the cell's own
// ranges of kslot and sortbuf (both unused by any other cell).  Returns the
// buffer holding the result.
__device__ __forceinline__ const unsigned long long *sort_large_cell(const FrameBuffers &b, uint32_t s, uint32_t n,
                                                     unsigned long long *sk) {
    const uint32_t tid = threadIdx.x;
    unsigned long long *a = reinterpret_cast<unsigned long long *>(b.kslot) + s;
    unsigned long long *t = b.sortbuf + s;
    for (uint32_t base = 0; base < n; base += kLdsSort) {
        const uint32_t len = min((uint32_t)kLdsSort, n - base);
        for (uint32_t i = tid; i < (uint32_t)kLdsSort; i += kCollideBlock)
            sk[i] = i < len ? ((unsigned long long)(b.src[s + base + i] & kSrcMask) << 32) | (base + i)
                            : ~0ull;
        __syncthreads();
        bitonic_lds(sk, kLdsSort);
        for (uint32_t i = tid; i < len; i += kCollideBlock) a[base + i] = sk[i];
        __syncthreads();
    }
    unsigned long long *from = a, *to = t;
    for (uint64_t w = kLdsSort; w < n; w *= 2) {
        for (uint64_t lo = 0; lo < n; lo += 2 * w) {
            const uint64_t mid = lo + w < n ? lo + w : n;
            const uint64_t hi = lo + 2 * w < n ? lo + 2 * w : n;
            merge_block(from + lo, (uint32_t)(mid - lo), from + mid, (uint32_t)(hi - mid), to + lo);
        }
        __syncthreads();
        unsigned long long *sw = from;
        from = to;
        to = sw;
    }
    return from;
}

template <int G>
__device__ __forceinline__ void collide_group(float &x, float &y, uint32_t r, uint32_t m,
                                              uint32_t gbase);

template <bool STEP>
__device__ __forceinline__ void big_cell(const FrameParams &p, const FrameBuffers &b, uint32_t s,
                                         uint32_t n, uint32_t c, unsigned long long *sk) {
    const uint32_t tid = threadIdx.x;
    const unsigned long long *perm;
    if (n <= (uint32_t)kLdsSort) {
        uint32_t P = 2;
        while (P < n) P <<= 1;
        for (uint32_t i = tid; i < P; i += kCollideBlock)
            sk[i] = i < n ? ((unsigned long long)(b.src[s + i] & kSrcMask) << 32) | i : ~0ull;
        __syncthreads();
        bitonic_lds(sk, P);
        perm = sk;
    } else {
        perm = sort_large_cell(b, s, n, sk);
    }
    if (STEP) {
        // Pass 1 over 256-rank chunks in canonical order: finish, write at
        // s + r, and rank each particle among the cell's particles going the
        // same way (ballots per wave, offsets across the block's waves, running
        // totals across chunks).  Ranks 0..8 are separated first by lanes
        // 0..8 of wave 0 (collide_group).  Per rank, `tmp` keeps (direction,
        // rank in it), or for a farther mover (key | bit 31, its slot); it is
        // whichever of kslot / sortbuf does not hold the order.
        __shared__ uint32_t s_wcnt[kWavesPerBlock][9], s_run[9], s_base[9];
        const uint32_t lane = tid & 63, wave = tid >> 6;
        const unsigned long long lt = lanemask_lt();
        const Grid g = grid_of(p, c);
        uint32_t cx, cy;
        cell_coords(g, c, cx, cy);
        uint2 *tmp = reinterpret_cast<const void *>(perm) == reinterpret_cast<const void *>(b.kslot + s)
                         ? reinterpret_cast<uint2 *>(b.sortbuf + s)
                         : b.kslot + s;
        if (tid < 9) s_run[tid] = 0;
        for (uint32_t base = 0; base < n; base += kCollideBlock) {
            const uint32_t r = base + tid;
            float2 q = make_float2(0.0f, 0.0f), v = make_float2(0.0f, 0.0f);
            if (r < n) {
                const uint32_t a = (uint32_t)perm[r];
                q = b.pos[s + a];
                v = b.vel[s + a];
            }
            if (base == 0 && wave == 0) collide_group<64>(q.x, q.y, lane, kMaxInCell, 0);
            uint32_t dir = 10, key = 0;
            if (r < n) {
                finish_particle(p, g, q.x, q.y, v.x, v.y);
                b.pos_out[s + r] = q;
                b.vel_out[s + r] = v;
                dir = direction(p, g, q.x, q.y, cx, cy, key);
            }
            uint32_t rin = 0;
#pragma unroll
            for (int d = 0; d < 9; ++d) {
                const unsigned long long m = __ballot(dir == (uint32_t)d);
                if (dir == (uint32_t)d) rin = (uint32_t)__popcll(m & lt);
                if (lane == 0) s_wcnt[wave][d] = (uint32_t)__popcll(m);
            }
            __syncthreads();
            if (dir < 9) {
                uint32_t off = s_run[dir];
                for (uint32_t w = 0; w < wave; ++w) off += s_wcnt[w][dir];
                tmp[r] = make_uint2(dir, off + rin);
            } else if (dir == 9) {
                const uint32_t slot = claim(b, key, 1u);
                tmp[r] = make_uint2(key | kRunFlag, slot | kRunFlag);
            }
            __syncthreads();
            if (tid < 9) {
                uint32_t t = 0;
                for (uint32_t w = 0; w < (uint32_t)kWavesPerBlock; ++w) t += s_wcnt[w][tid];
                s_run[tid] += t;
            }
            __syncthreads();
        }
        // One atomic per occupied direction, then the slots.
        if (tid < 9) {
            const uint32_t tx = cx + tid % 3 - 1, ty = cy + tid / 3 - 1;
            s_base[tid] = s_run[tid] ? claim(b, g.base + ty * g.gx + tx, s_run[tid]) : 0u;
        }
        __syncthreads();
        for (uint32_t r = tid; r < n; r += kCollideBlock) {
            const uint2 t = tmp[r];
            if (t.x & kRunFlag) {
                b.kslot[s + r] = make_uint2(t.x & kSrcMask, t.y);
            } else {
                const uint32_t key = g.base + (cy + t.x / 3 - 1) * g.gx + (cx + t.x % 3 - 1);
                b.kslot[s + r] = make_uint2(key, (s_base[t.x] + t.y) | (t.y == 0 ? kRunFlag : 0u));
            }
        }
    } else {
        for (uint32_t r = tid; r < n; r += kCollideBlock) {
            const uint32_t a = (uint32_t)perm[r];
            b.pos_out[s + r] = b.pos[s + a];
            b.vel_out[s + r] = b.vel[s + a];
        }
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// The collide pass.

// Size class of a queued cell of n particles (kClasses for none: 0 or 1
// particle).  For 2 <= n <= 64 the class is ceil(log2(n)) - 1.
__device__ __forceinline__ uint32_t size_class(uint32_t n) {
    if (n < 2) return (uint32_t)kClasses;
    if (n > kWideMax) return (uint32_t)kBlockClass;
    const uint32_t k = 31u - (uint32_t)__builtin_clz(n - 1);
    return k < (uint32_t)kWaveClass ? k : (uint32_t)kWaveClass;
}

// Wave-private LDS of a cell wave of the wide path (below).
constexpr int kWideRuns = 256;  // runs per cell ordered by runs (more: pairwise ranks)
struct WaveLds {
    uint32_t code[kWideMax];          // per rank >= 9: direction (bit 31 set); 0 for a far mover
    uint32_t head_key[kWideRuns];     // first source index of each run
    uint32_t head_pos[kWideRuns];     // stored position of each run's start
    uint32_t run_off[kWideRuns];      // canonical rank of each run's start minus its position
    uint2 head_kl[kWideRuns];         // (first source index, length) of each run
    uint2 dir_tbl[9];                 // per direction: (new cell key, first slot)
};

// Gauss-Seidel on the first m = min(n, 9) particles of a cell held by lanes
// gbase + r (r = canonical rank).  In the in-order loop (particles.rs:62-81)
// pair (i,j) can run at step i + j: the pairs of one step touch disjoint
// particles and every particle still sees its updates in the loop's order, so
// 2M - 3 steps (M = min(G, 9)) give the loop's result bit for bit.  Both lanes
// of a pair fetch the other's position and evaluate collide_pair's arithmetic
// on the same operands; the lower rank applies -dv, the higher +dv.  All
// lanes execute the shuffles.
// Step t of that schedule for the lane holding rank ri of a cell whose
// first mi ranks collide, ranks held by lanes gbase + r.  The pair rule is
// Particles::pairs (particles.rs:65-92): glam distance, skip beyond
// MIN_DISTANCE = 1, 0 -> 0.0001, force (0.5*(1-d))/d, equal and opposite
// displacement.
__device__ __forceinline__ void separate_step(float &x, float &y, int ri, int mi, int gbase, int t) {
    const int lane = (int)lane_id();
    const int partner = t - ri;
    const bool left = ri < partner && partner < mi;
    const bool right = partner >= 0 && partner < ri && ri < mi;
    const int from = (left || right) ? gbase + partner : lane;
    const float qx = __shfl(x, from, 64);
    const float qy = __shfl(y, from, 64);
    if (left || right) {
        const float xi = left ? x : qx, yi = left ? y : qy;
        const float xj = left ? qx : x, yj = left ? qy : y;
        const float dx = xi - xj;
        const float dy = yi - yj;
        float sq = dx * dx;
        sq = sq + dy * dy;
        float d = sqrtf(sq);
        if (!(d > 1.0f)) {
            if (d == 0.0f) d = 0.0001f;
            const float f = (0.5f * (1.0f - d)) / d;
            const float ex = (xj - xi) * f;
            const float ey = (yj - yi) * f;
            if (left) {
                x = x - ex;
                y = y - ey;
            } else {
                x = x + ex;
                y = y + ey;
            }
        }
    }
}

template <int G>
__device__ __forceinline__ void collide_group(float &x, float &y, uint32_t r, uint32_t m,
                                              uint32_t gbase) {
    constexpr int M = G < kMaxInCell ? G : kMaxInCell;
#pragma unroll
    for (int t = 1; t <= 2 * M - 3; ++t) separate_step(x, y, (int)r, (int)m, (int)gbase, t);
}

// ---------------------------------------------------------------------------
// collide_kernel: one packed particle per lane, the 64 consecutive particles
// i0 .. i0 + 63 per wavefront, whose cells come from `key` (written by the
// previous frame's scatter or by the upload): a cell is a segment of equal
// keys.
//  - A cell of at most kInWaveMax particles that lies inside the wavefront is
//    handled there, with the arithmetic of the cell kernels' lane groups:
//    ranked by source index, moved to lane (first lane + rank), separated,
//    finished and written at i0 + lane (its canonical index), slots claimed
//    with one atomic per direction.  The wavefront reads whole lines of pos,
//    vel, src and key and writes whole lines of pos_out, vel_out and kslot;
//    before the collapse under gravity almost every cell is such a segment.
//    Every lane runs the separation steps of the wavefront's largest such
//    cell, so the cap bounds them (2 * 3 - 3 = 3 steps); larger cells go to
//    the lane groups of cells_kernel, which are sorted by size.
//  - Any other cell whose first particle lies in the wavefront -- larger, or
//    running past the wavefront's last particle -- is queued by size class
//    for cells_kernel, with its range from the offsets.  The range must start
//    at that particle and agree with the keys, or the kernel raises
//    kErrLayout and queues nothing for it (keys and offsets that disagree
//    would make queued ranges overlap).
//  - The lanes of a cell that began before the wavefront leave it to the
//    wavefront that queued it.  The kernel has no barrier: a wavefront with
//    nothing to handle or queue returns after the keys, and queued cells go
//    to their lists with one atomic each (slice = wavefront % kSlices).
constexpr uint32_t kInWaveMax = 3;

// Reductions of a wavefront into lane 63 by DPP moves (one instruction a
// step; a shuffle takes three): lanes without a source add or compare 0.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp0(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}

__device__ __forceinline__ uint32_t wave63_max(uint32_t v) {
    v = max(v, dpp0<0x111, 0xf>(v));  // row_shr:1, :2, :4, :8
    v = max(v, dpp0<0x112, 0xf>(v));
    v = max(v, dpp0<0x114, 0xf>(v));
    v = max(v, dpp0<0x118, 0xf>(v));
    v = max(v, dpp0<0x142, 0xa>(v));  // row_bcast:15 into rows 1 and 3
    return max(v, dpp0<0x143, 0xc>(v));  // row_bcast:31 into rows 2 and 3
}

// The wavefront's largest value, in every lane (a scalar).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    return __builtin_amdgcn_readlane(wave63_max(v), 63);
}

// The value of the lane before, of the lane after; lane 0's and lane 63's:
// `edge`.  With these and the maximum as DPP moves instead of shuffles through
// LDS the collide kernel takes 13.0 us on the 1M lattice (13.4) and 82.8 on
// the 4M blobs (84.4), the canonical order of 1M particles 12.3 (12.9).
__device__ __forceinline__ uint32_t from_lane_before(uint32_t v, uint32_t edge) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)edge, (int)v, 0x138, 0xf, 0xf, false);  // wave_shr:1
}

__device__ __forceinline__ uint32_t from_lane_after(uint32_t v, uint32_t edge) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)edge, (int)v, 0x130, 0xf, 0xf, false);  // wave_shl:1
}

// Start and end of cell k (k < ncell) as cell_start gives them, the six
// loads in flight together.
__device__ __forceinline__ void cell_range(const FrameParams &p, const FrameBuffers &b, uint32_t k,
                                           uint32_t &st, uint32_t &en) {
    const uint32_t c0 = k >> kChunkShift;
    const uint32_t live0 = b.chunk_live[c0], w0 = offset_word(b, k), pre0 = b.chunk_prefix[c0];
    const bool last = k + 1 >= p.ncell;
    const uint32_t k1 = last ? k : k + 1, c1 = k1 >> kChunkShift;
    const uint32_t live1 = b.chunk_live[c1], w1 = offset_word(b, k1), pre1 = b.chunk_prefix[c1];
    uint32_t at0 = offset_entry(b, k, w0), at1 = offset_entry(b, k1, w1);
    if (b.off_shift) {
        at0 = wide_entry(b, k, at0, live0);
        at1 = wide_entry(b, k1, at1, live1);
    }
    st = offset_of(at0, live0, pre0);
    en = last ? p.n : offset_of(at1, live1, pre1);
    st = st < p.n ? st : p.n;
    en = en < p.n ? en : p.n;
}

// 64-particle windows per wavefront (the kernel takes any number: each
// window's loads and slot atomics are in flight together).  One is the
// fastest measured: with 2..4 the frame before the collapse is no faster and
// the collapsed frame is slower.
constexpr int kCollideWindows = 1;

__global__ __launch_bounds__(kCollideBlock) void collide_kernel(FrameParams p, FrameBuffers b) {
    constexpr int W = kCollideWindows;
    const uint32_t lane = lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t base = (blockIdx.x * kWavesPerBlock + wave) * (64u * W);
    uint32_t k[W];
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const uint32_t i = base + 64u * j + lane;
        k[j] = i < p.n ? b.key[i] : kNoKey;
    }
    // The keys on either side of the wavefront's particles: lane 0 reads the
    // one before, lane 63 the one after.
    uint32_t before = kNoKey, after = kNoKey;
    if (lane == 0 && base > 0 && base < p.n) before = b.key[base - 1];
    if (lane == 63 && base + 64u * W < p.n) after = b.key[base + 64u * W];
    // A frame after one that raised an error (a scan that gave up its
    // look-back, keys that disagree with the offsets) reads no offsets: the
    // context is dead.  A vector load beside the keys (no barrier follows in
    // this kernel, so wavefronts need not agree).
    const uint32_t dead = b.error[lane >> 6];
    before = __builtin_amdgcn_readlane(before, 0);
    after = __builtin_amdgcn_readlane(after, 63);

    // Per window: my cell's first and last lane (tl == 64: past the window),
    // whether this window handles it (mine) or queues it (queue).
    int hl[W], tl[W];
    uint32_t m[W];
    bool mine[W], queue[W];
    bool work = false, bad = false;
    const unsigned long long lt = lanemask_lt(), le = lt | (1ull << lane);
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const uint32_t i = base + 64u * j + lane;
        const bool valid = i < p.n;
        const uint32_t wb = j == 0 ? before : __builtin_amdgcn_readlane(k[j > 0 ? j - 1 : 0], 63);
        const uint32_t wa = j == W - 1 ? after : __builtin_amdgcn_readlane(k[j < W - 1 ? j + 1 : 0], 0);
        const uint32_t kp = from_lane_before(k[j], wb), kn = from_lane_after(k[j], wa);
        const bool head = valid && k[j] != kp;
        const bool tail = valid && k[j] != kn;
        const unsigned long long heads = __ballot(head), tails = __ballot(tail);
        const unsigned long long hb = heads & le, ta = tails & ~lt;
        hl[j] = hb ? 63 - (int)__builtin_clzll(hb) : -1;
        tl[j] = ta ? (int)__builtin_ctzll(ta) : 64;
        // A key past the grid is a layout no upload or frame writes.
        const bool kbad = valid && k[j] >= p.ncell;
        const bool inside = valid && !kbad && hl[j] >= 0 && tl[j] < 64;
        m[j] = inside ? (uint32_t)(tl[j] - hl[j] + 1) : 0u;
        mine[j] = inside && m[j] <= kInWaveMax;
        queue[j] = head && !kbad && !mine[j];
        work = work || mine[j] || queue[j];
        bad = bad || kbad;
    }
    if (__builtin_amdgcn_readfirstlane(dead)) return;
    if (bad) raise_error(b, kErrLayout);
    if (__ballot(work) == 0) return;  // every lane votes; nothing to handle or queue

    // Loads: the queued cells' ranges and the handled particles, all windows.
    uint32_t qst[W], qen[W], sv[W];
    float2 q[W], w[W];
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const uint32_t i = base + 64u * j + lane;
        qst[j] = qen[j] = 0;
        if (queue[j]) cell_range(p, b, k[j], qst[j], qen[j]);
        sv[j] = 0;
        q[j] = w[j] = make_float2(0.0f, 0.0f);
        if (mine[j]) {
            sv[j] = b.src[i] & kSrcMask;
            q[j] = b.pos[i];
            w[j] = b.vel[i];
        }
    }

    // The first particle of a cell this window does not handle queues it.
    uint32_t cls[W], qs[W], qn[W];
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const uint32_t i = base + 64u * j + lane;
        const uint32_t i0 = base + 64u * j;
        cls[j] = (uint32_t)kClasses;
        qs[j] = qn[j] = 0;
        if (queue[j]) {
            const bool ok = tl[j] == 64 ? qen[j] >= i0 + 64 : qen[j] == i0 + (uint32_t)tl[j] + 1;
            if (qst[j] == i && ok && qen[j] <= p.n) {
                qs[j] = qst[j];
                qn[j] = qen[j] - qst[j];
                cls[j] = size_class(qn[j]);
            } else {
                raise_error(b, kErrLayout);
            }
        }
    }

    // Handled cells: rank, separate, finish, claim (every window's atomics
    // in flight together), then write.
    uint32_t nkey[W], rin[W], leader[W], got[W];
    bool near[W];
    float px[W], py[W], vx[W], vy[W];
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const uint32_t mw = wave_max_u32(mine[j] ? m[j] : 0u);
        // Canonical rank: source indices inside a cell are distinct.
        uint32_t rank = 0;
        for (uint32_t t = 0; t < mw; ++t) {
            const bool in = mine[j] && t < m[j];
            const uint32_t o = (uint32_t)__shfl((int)sv[j], in ? hl[j] + (int)t : (int)lane, 64);
            rank += (in && o < sv[j]) ? 1u : 0u;
        }
        const int to = (mine[j] ? hl[j] + (int)rank : (int)lane) * 4;
        px[j] = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(q[j].x)));
        py[j] = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(q[j].y)));
        vx[j] = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(w[j].x)));
        vy[j] = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(w[j].y)));
        // Lane hl + r now holds rank r of its cell (m <= kInWaveMax < 9: every
        // rank collides).
        const int r = mine[j] ? (int)lane - hl[j] : 0;
        const int mi = mine[j] ? (int)m[j] : 0;
        for (int t = 1; t <= 2 * (int)mw - 3; ++t) separate_step(px[j], py[j], r, mi, mine[j] ? hl[j] : 0, t);

        uint32_t dir = 10;
        nkey[j] = 0;
        if (mine[j]) {
            const Grid g = grid_of(p, k[j]);
            uint32_t cx, cy;
            cell_coords(g, k[j], cx, cy);
            finish_particle(p, g, px[j], py[j], vx[j], vy[j]);
            dir = direction(p, g, px[j], py[j], cx, cy, nkey[j]);
        }
        // Lanes of my cell going the same way.
        unsigned long long same = 0;
#pragma unroll
        for (int d = 0; d < 9; ++d) {
            const unsigned long long bm = __ballot(dir == (uint32_t)d);
            same = dir == (uint32_t)d ? bm : same;
        }
        const unsigned long long upto = tl[j] >= 63 ? ~0ull : (1ull << (tl[j] + 1)) - 1;
        const unsigned long long seg = mine[j] ? upto & ~((1ull << hl[j]) - 1) : 0ull;
        same &= seg;
        near[j] = dir < 9;
        rin[j] = (uint32_t)__popcll(same & lt);
        leader[j] = near[j] ? (uint32_t)__builtin_ctzll(same) : lane;
        got[j] = 0;
        if (mine[j] && (!near[j] || rin[j] == 0))
            got[j] = claim(b, nkey[j], near[j] ? (uint32_t)__popcll(same) : 1u);
    }
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const uint32_t i = base + 64u * j + lane;
        const uint32_t first = (uint32_t)__shfl((int)got[j], (int)leader[j], 64);
        if (mine[j]) {
            const uint32_t slot = near[j] ? (first + rin[j]) | (rin[j] == 0 ? kRunFlag : 0u) : (got[j] | kRunFlag);
            b.pos_out[i] = make_float2(px[j], py[j]);
            b.vel_out[i] = make_float2(vx[j], vy[j]);
            b.kslot[i] = make_uint2(nkey[j], slot);
        }
    }

    // Queued cells, one global atomic each into slice (wavefront % kSlices)
    // of their class; what does not fit goes to the class's overflow list.
    const uint32_t slice = (blockIdx.x * kWavesPerBlock + wave) % kSlices;
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const uint32_t c = cls[j];
        if (c < (uint32_t)kClasses) {
            const uint4 ent = make_uint4(qs[j], qn[j], k[j], 0);
            const uint32_t a = atomicAdd(&b.class_ctr[ctr_index((int)c, slice)], 1u);
            if (a < b.slice_cap[c]) {
                b.cells[b.class_off[c] + slice * b.slice_cap[c] + a] = ent;
            } else {
                const uint32_t o = atomicAdd(&b.class_ctr[ctr_index((int)c, kSlices)], 1u);
                if (o < b.class_cap[c]) b.cells[b.class_off[c] + kSlices * b.slice_cap[c] + o] = ent;
            }
        }
    }
}

// Cells of 2 <= n <= G particles (G = 2..64), 64 / G cells per wavefront,
// one particle per lane.  Each group of G lanes:
//  1. loads its cell's particles (lane j: stored position j);
//  2. ranks them by source index (the canonical order) and moves rank r to
//     lane gbase + r;
//  3. hands them to ranked_group (below).
template <int G>
__device__ __forceinline__ void ranked_group(const FrameParams &p, const FrameBuffers &b,
                                             float px, float py, float vx, float vy, uint32_t j,
                                             uint32_t n, uint32_t s, uint32_t c, uint32_t gbase);

// One lane's share of a group item: its cell (s, n, c) and, in lane j of
// the group, stored particle j.  group_load issues the loads; group_run
// waits for them, so a wavefront can load its next item while it computes.
struct GroupItem {
    uint32_t s, n, c, key;
    float2 q, w;
};

template <int G>
__device__ __forceinline__ uint4 group_entry(const uint4 *list, uint32_t count) {
    const uint32_t e = lane_id() / G;
    return e < count ? list[e] : make_uint4(0, 0, 0, 0);
}

template <int G>
__device__ __forceinline__ GroupItem group_load(const FrameBuffers &b, uint4 cell) {
    const uint32_t j = lane_id() % G;
    GroupItem it;
    it.s = cell.x;
    it.n = cell.y;
    it.c = cell.z;
    it.key = 0xffffffffu;
    it.q = it.w = make_float2(0.0f, 0.0f);
    if (j < it.n) {
        it.key = b.src[it.s + j] & kSrcMask;
        it.q = b.pos[it.s + j];
        it.w = b.vel[it.s + j];
    }
    return it;
}

template <int G>
__device__ __forceinline__ void group_run(const FrameParams &p, const FrameBuffers &b,
                                          const GroupItem &it) {
    const uint32_t lane = lane_id();
    const uint32_t j = lane % G;
    const uint32_t gbase = lane - j;
    const uint32_t s = it.s, n = it.n, c = it.c, key = it.key;
    const float2 q = it.q, w = it.w;
    // Source indices inside a cell are distinct; empty lanes keep their own
    // position after the n particles.
    uint32_t rank = 0;
#pragma unroll
    for (int k = 0; k < G; ++k) rank += __shfl(key, (int)gbase + k, 64) < key;
    if (j >= n) rank = j;
    const int to = (int)(gbase + rank) * 4;
    float px = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(q.x)));
    float py = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(q.y)));
    float vx = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(w.x)));
    float vy = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(w.y)));

    // Lane gbase + r now holds rank r.
    ranked_group<G>(p, b, px, py, vx, vy, j, n, s, c, gbase);
}

// The particles of ranks 0..n-1 of a cell segment that starts at canonical
// index s, held by lanes gbase + r of a group of G lanes: separate the first
// min(n, 9) (collide_group), finish every particle, write it at s + r, and
// claim slots: one atomic per occupied neighbour direction (by the
// direction's first lane) reserves a run of consecutive slots in canonical
// order; a farther mover takes a slot of its own.
template <int G>
__device__ __forceinline__ void ranked_group(const FrameParams &p, const FrameBuffers &b,
                                             float px, float py, float vx, float vy, uint32_t j,
                                             uint32_t n, uint32_t s, uint32_t c, uint32_t gbase) {
    const uint32_t lane = lane_id();
    collide_group<G>(px, py, j, n < (uint32_t)kMaxInCell ? n : (uint32_t)kMaxInCell, gbase);

    const bool has = j < n;
    const Grid g = grid_of(p, c);
    uint32_t cx, cy;
    cell_coords(g, c, cx, cy);
    uint32_t dir = 10, nkey = 0;
    if (has) {
        finish_particle(p, g, px, py, vx, vy);
        dir = direction(p, g, px, py, cx, cy, nkey);
        b.pos_out[s + j] = make_float2(px, py);
        b.vel_out[s + j] = make_float2(vx, vy);
    }
    // Lanes of this group going the same way.
    unsigned long long same = 0;
#pragma unroll
    for (int d = 0; d < 9; ++d) {
        const unsigned long long m = __ballot(dir == (uint32_t)d);
        same = dir == (uint32_t)d ? m : same;
    }
    const unsigned long long gmask = G == 64 ? ~0ull : (((1ull << G) - 1) << gbase);
    same &= gmask;
    const bool near = dir < 9;
    const uint32_t rin = (uint32_t)__popcll(same & lanemask_lt());
    const uint32_t leader = near ? (uint32_t)__builtin_ctzll(same) : lane;
    uint32_t got = 0;
    if (has && (!near || rin == 0))
        got = claim(b, nkey, near ? (uint32_t)__popcll(same) : 1u);
    const uint32_t base = (uint32_t)__shfl((int)got, (int)leader, 64);
    if (has) {
        const uint32_t slot = near ? (base + rin) | (rin == 0 ? kRunFlag : 0u) : (got | kRunFlag);
        b.kslot[s + j] = make_uint2(nkey, slot);
    }
}

// ---------------------------------------------------------------------------
// Cells of 65..kWideChunks*64 particles, three per block: waves 0..2 take one
// cell each, wave 3 separates the first nine particles of all three.
//
// Ranks 0..8 and ranks 9..n-1 of a cell claim their slots independently, each
// direction's share of either part as its own run.  Both runs are ascending
// in canonical index and every index of the first lies below every index of
// the second, so in the new cell they are two runs that do not interleave,
// which is all the order restoration of the next frame needs.  The cell
// waves therefore never wait for the Gauss-Seidel chain.

constexpr int kWideCells = kWavesPerBlock - 1;

struct WideStage {
    float4 q[kWideCells][kMaxInCell];  // ranks 0..8 of each cell: x, y, stored position (bits)
    float2 v[kWideCells][kMaxInCell];  // and their velocities
    uint2 sc[kWideCells];              // each cell's first particle and key
    uint32_t on[kWideCells];           // nonzero: wave 3 handles ranks 0..8
};

// Cell wave, before the block barrier: loads in stored order, canonical rank
// of every stored position (rk), ranks 0..8 (position, stored position and
// velocity) staged for wave 3.  The ranks
// come from the runs; a cell of more than kWideRuns runs is ranked pairwise
// (source indices in a cell are distinct).
__device__ __forceinline__ void wide_order(const FrameBuffers &b, uint32_t s, uint32_t n,
                                           WaveLds &L, float4 *stage, float2 *vstage,
                                           float2 (&pp)[kWideChunks],
                                           float2 (&vv)[kWideChunks],
                                           uint32_t (&rk)[kWideChunks]) {
    const uint32_t lane = lane_id();
    const unsigned long long le = lanemask_lt() | (1ull << lane);
    uint32_t sv[kWideChunks];
#pragma unroll
    for (int q = 0; q < kWideChunks; ++q) {
        const uint32_t i = 64 * q + lane;
        sv[q] = 0;
        pp[q] = vv[q] = make_float2(0.0f, 0.0f);
        if (i < n) {
            sv[q] = b.src[s + i];
            pp[q] = b.pos[s + i];
            vv[q] = b.vel[s + i];
        }
    }
    // Runs: flagged particles and position 0 start one.
    uint32_t runs = 0, rid[kWideChunks];
#pragma unroll
    for (int q = 0; q < kWideChunks; ++q) {
        const uint32_t i = 64 * q + lane;
        const bool start = i < n && (i == 0 || (sv[q] & kRunFlag));
        const unsigned long long m = __ballot(start);
        rid[q] = runs + (uint32_t)__popcll(m & le) - 1;
        if (start && rid[q] < (uint32_t)kWideRuns) {
            L.head_key[rid[q]] = sv[q] & kSrcMask;
            L.head_pos[rid[q]] = i;
        }
        runs += (uint32_t)__popcll(m);
    }
    if (runs <= (uint32_t)kWideRuns) {
        wave_sync();
        // Lane l owns runs l, l + 64, ...
        constexpr int kOwn = kWideRuns / 64;
#pragma unroll
        for (int k = 0; k < kOwn; ++k) {
            const uint32_t r = lane + 64 * k;
            if (r < runs) {
                const uint32_t end = r + 1 < runs ? L.head_pos[r + 1] : n;
                L.head_kl[r] = make_uint2(L.head_key[r], end - L.head_pos[r]);
            }
        }
        wave_sync();
        // Canonical rank of a run's start: particles in runs with a smaller
        // first source index.  Stored as rank - position so that
        // rank = run_off + i.
        uint32_t hk[kOwn], off[kOwn];
#pragma unroll
        for (int k = 0; k < kOwn; ++k) {
            const uint32_t r = lane + 64 * k;
            hk[k] = r < runs ? L.head_key[r] : 0u;
            off[k] = 0;
        }
        if (runs <= 64) {  // the common case: one run per lane at most
#pragma unroll 4
            for (uint32_t j = 0; j < runs; ++j) {
                const uint2 e = L.head_kl[j];
                off[0] += e.x < hk[0] ? e.y : 0u;
            }
        } else {
#pragma unroll 2
            for (uint32_t j = 0; j < runs; ++j) {
                const uint2 e = L.head_kl[j];
#pragma unroll
                for (int k = 0; k < kOwn; ++k) off[k] += e.x < hk[k] ? e.y : 0u;
            }
        }
#pragma unroll
        for (int k = 0; k < kOwn; ++k) {
            const uint32_t r = lane + 64 * k;
            if (r < runs) L.run_off[r] = off[k] - L.head_pos[r];
        }
        wave_sync();
#pragma unroll
        for (int q = 0; q < kWideChunks; ++q) {
            const uint32_t i = 64 * q + lane;
            rk[q] = i < n ? L.run_off[rid[q]] + i : 0xffffffffu;
        }
    } else {
        // Pairwise: rank = number of smaller source indices (code[] is free
        // until after the block barrier).
        wave_sync();
#pragma unroll
        for (int q = 0; q < kWideChunks; ++q) {
            const uint32_t i = 64 * q + lane;
            if (i < n) L.code[i] = sv[q] & kSrcMask;
            rk[q] = 0;
        }
        wave_sync();
        for (uint32_t j = 0; j < n; ++j) {
            const uint32_t o = L.code[j];
#pragma unroll
            for (int q = 0; q < kWideChunks; ++q) rk[q] += o < (sv[q] & kSrcMask);
        }
#pragma unroll
        for (int q = 0; q < kWideChunks; ++q)
            if (64 * q + lane >= n) rk[q] = 0xffffffffu;
    }
#pragma unroll
    for (int q = 0; q < kWideChunks; ++q) {
        const uint32_t i = 64 * q + lane;
        if (i < n && rk[q] < (uint32_t)kMaxInCell) {
            stage[rk[q]] = make_float4(pp[q].x, pp[q].y, __uint_as_float(i), 0.0f);
            vstage[rk[q]] = vv[q];
        }
    }
}

// Cell wave, after the barrier: ranks 9..n-1.  Finish in stored order, write
// at s + rank, keep each rank's direction (or a far mover's key) in LDS; then
// in canonical order count per direction, one atomic per occupied direction,
// and the slots.
__device__ __forceinline__ void wide_rest(const FrameParams &p, const FrameBuffers &b, uint32_t s,
                                          uint32_t n, uint32_t c, WaveLds &L,
                                          const float2 (&pp)[kWideChunks],
                                          const float2 (&vv)[kWideChunks],
                                          const uint32_t (&rk)[kWideChunks]) {
    const uint32_t lane = lane_id();
    const unsigned long long lt = lanemask_lt();
    const Grid g = grid_of(p, c);
    uint32_t cx, cy;
    cell_coords(g, c, cx, cy);
    uint32_t *code = L.code;
    uint32_t fkey[kWideChunks];  // a farther mover's new key, or ~0
#pragma unroll
    for (int q = 0; q < kWideChunks; ++q) {
        fkey[q] = 0xffffffffu;
        // rk is ~0 past the particles: one compare covers both bounds.
        if (rk[q] - (uint32_t)kMaxInCell < n - (uint32_t)kMaxInCell) {
            float px = pp[q].x, py = pp[q].y, vx = vv[q].x, vy = vv[q].y;
            finish_particle(p, g, px, py, vx, vy);
            b.pos_out[s + rk[q]] = make_float2(px, py);
            b.vel_out[s + rk[q]] = make_float2(vx, vy);
            uint32_t key;
            const uint32_t dir = direction(p, g, px, py, cx, cy, key);
            code[rk[q]] = dir < 9 ? (kRunFlag | (dir << 27)) : 0u;
            if (dir == 9) fkey[q] = key;
        }
    }
    wave_sync();
    // Canonical order, chunk by chunk: each near mover's rank in its
    // direction, written back into code[] (a rolled loop keeps the ballot
    // masks of one chunk live at a time).
    uint32_t count[9];
#pragma unroll
    for (int d = 0; d < 9; ++d) count[d] = 0;
    uint32_t next = kMaxInCell + lane < n ? code[kMaxInCell + lane] : 0u;
#pragma unroll 1
    for (uint32_t r0 = kMaxInCell; r0 < n; r0 += 64) {
        const uint32_t r = r0 + lane;
        const uint32_t w = next;
        next = r + 64 < n ? code[r + 64] : 0u;
        const uint32_t dir = (w & kRunFlag) ? (w >> 27) & 15u : 10u;
        uint32_t rin = 0;
#pragma unroll
        for (int d = 0; d < 9; ++d) {
            const unsigned long long m = __ballot(dir == (uint32_t)d);
            if (dir == (uint32_t)d) rin = count[d] + (uint32_t)__popcll(m & lt);
            count[d] += (uint32_t)__popcll(m);
        }
        if (dir < 9) code[r] = kRunFlag | (dir << 27) | rin;
    }
    // Every atomic of the cell in one round: one per occupied direction
    // (lanes 0..8), one per farther mover.
    uint32_t mine = 0;
#pragma unroll
    for (int d = 0; d < 9; ++d) mine = lane == (uint32_t)d ? count[d] : mine;
    uint32_t got = 0, tkey = 0;
    if (lane < 9) {
        const uint32_t tx = cx + lane % 3 - 1, ty = cy + lane / 3 - 1;
        tkey = g.base + ty * g.gx + tx;
        if (mine > 0) got = claim(b, tkey, mine);
    }
    uint32_t fslot[kWideChunks];
#pragma unroll
    for (int q = 0; q < kWideChunks; ++q)
        fslot[q] = fkey[q] != 0xffffffffu ? claim(b, fkey[q], 1u) : 0u;
    // Per direction: (new key, first slot), then the slots.
    if (lane < 9) L.dir_tbl[lane] = make_uint2(tkey, got);
    wave_sync();
#pragma unroll 1
    for (uint32_t r0 = kMaxInCell; r0 < n; r0 += 64) {
        const uint32_t r = r0 + lane;
        const uint32_t w = r < n ? code[r] : 0u;
        if (w & kRunFlag) {
            const uint32_t rin = w & 0x07ffffffu;
            const uint2 t = L.dir_tbl[(w >> 27) & 15u];
            b.kslot[s + r] = make_uint2(t.x, (t.y + rin) | (rin == 0 ? kRunFlag : 0u));
        }
    }
#pragma unroll
    for (int q = 0; q < kWideChunks; ++q)
        if (fkey[q] != 0xffffffffu) b.kslot[s + rk[q]] = make_uint2(fkey[q], fslot[q] | kRunFlag);
}

// One block item: cells list[0..2], of which `count` exist.
__device__ __forceinline__ void wide_item(const FrameParams &p, const FrameBuffers &b,
                                          const uint4 *list, uint32_t count, WaveLds *lds,
                                          WideStage &st) {
    // readfirstlane: the compiler then knows the wave index is uniform and
    // branches on it instead of running both sides under lane masks.
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
    // Defined on every path, so that they are not carried around the item
    // loop (and kept live through wave 3's branch).
    float2 pp[kWideChunks], vv[kWideChunks];
    uint32_t rk[kWideChunks];
#pragma unroll
    for (int q = 0; q < kWideChunks; ++q) {
        pp[q] = vv[q] = make_float2(0.0f, 0.0f);
        rk[q] = 0;
    }
    uint4 cell = make_uint4(0, 0, 0, 0);
    bool mine = false, fast = false;
    __syncthreads();  // the previous item's stage has been read
    if (wave < (uint32_t)kWideCells) {
        const uint32_t e = wave;
        mine = e < count;
        if (mine) {
            cell = list[e];
            if (cell.y <= kWideMax) {  // always, by the class; guards a corrupt list
                wide_order(b, cell.x, cell.y, lds[wave], st.q[wave], st.v[wave], pp, vv, rk);
                fast = true;
            }
        }
        if (lane == 0) {
            st.on[wave] = fast ? 1u : 0u;
            st.sc[wave] = make_uint2(cell.x, cell.z);
        }
    }
    __syncthreads();
    if (wave == (uint32_t)kWideCells) {
        // Lanes 16g + j, j < 9: rank j of cell g.
        const uint32_t g = lane / 16, j = lane % 16;
        const uint32_t e = g;
        uint32_t s = 0, c = 0, m = 0;
        float4 q = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float2 v = make_float2(0.0f, 0.0f);
        if (g < (uint32_t)kWideCells && e < count && st.on[g]) {
            // The cell waves staged all of it: no global load before the
            // Gauss-Seidel chain.
            const uint2 sc = st.sc[g];
            s = sc.x;
            c = sc.y;
            m = kMaxInCell;
            if (j < (uint32_t)kMaxInCell) {
                q = st.q[g][j];
                v = st.v[g][j];
            }
        }
        ranked_group<16>(p, b, q.x, q.y, v.x, v.y, j, m, s, c, 16 * g);
    } else if (fast) {
        wide_rest(p, b, cell.x, cell.y, cell.z, lds[wave], pp, vv, rk);
    }
}

// Work items of the queued classes.  Class k's items take `per` cells each
// (64 / G for a group class, three for class 6, one for class 7) and are
// numbered slice by slice, then the overflow list.  ItemMap holds, per
// class, the inclusive prefix of items over the slices (in LDS), the slice
// fills and the totals.
struct ItemMap {
    uint32_t incl[kClasses][kSlices];
    uint32_t fill[kClasses][kSlices + 1];  // [kSlices]: the overflow list
    uint32_t in_slices[kClasses];          // items in the slices
    uint32_t items[kClasses];              // all items of the class
    uint32_t off[kClasses];                // class_off and slice_cap, kept here
    uint32_t scap[kClasses];               // rather than in scalar registers
};

__host__ __device__ constexpr uint32_t cells_per_item(int k) {
    return k < kGroupClasses ? (32u >> k) : k == kWaveClass ? (uint32_t)kWideCells : 1u;
}

// Fills the map: wave w takes classes w and w + 4, lane l slice l.  Every
// block waits for it before its first item, so both classes' counters, their
// overflow lists' too, are loaded together, and the sums are DPP moves.
__device__ __forceinline__ void build_item_map(const FrameBuffers &b, ItemMap &m) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
    uint32_t fill[2], over[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int k = (int)wave + 4 * h;
        fill[h] = b.class_ctr[ctr_index(k, (int)lane)];
        over[h] = b.class_ctr[ctr_index(k, kSlices)];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int k = (int)wave + 4 * h;
        // constant indices into the kernel-argument arrays (a variable index
        // would copy them to scratch memory)
        uint32_t scap = 0, ccap = 0, off = 0;
#pragma unroll
        for (int kk = 0; kk < kClasses; ++kk) {
            scap = k == kk ? b.slice_cap[kk] : scap;
            ccap = k == kk ? b.class_cap[kk] : ccap;
            off = k == kk ? b.class_off[kk] : off;
        }
        const uint32_t per = cells_per_item(k);
        const uint32_t f = min(fill[h], scap);
        const uint32_t incl = wave_inclusive_sum((f + per - 1) / per);
        m.incl[k][lane] = incl;
        m.fill[k][lane] = f;
        if (lane == 63) {
            const uint32_t fo = min(over[h], ccap);
            m.fill[k][kSlices] = fo;
            m.in_slices[k] = incl;
            m.items[k] = incl + (fo + per - 1) / per;
            m.off[k] = off;
            m.scap[k] = scap;
        }
    }
}

// Item v (below m.items[k], the same in every lane) of class k: its first
// cell and how many cells of its list segment start there.
__device__ __forceinline__ const uint4 *locate(const FrameBuffers &b, const ItemMap &m, int k,
                                               uint32_t v, uint32_t &avail) {
    const uint32_t per = cells_per_item(k);
    uint32_t seg, local;
    if (v < m.in_slices[k]) {
        seg = (uint32_t)__popcll(__ballot(m.incl[k][lane_id()] <= v));
        local = v - (seg ? m.incl[k][seg - 1] : 0u);
    } else {
        seg = kSlices;
        local = v - m.in_slices[k];
    }
    avail = m.fill[k][seg] - local * per;
    return b.cells + m.off[k] + seg * m.scap[k] + local * per;
}

// Work items [start, stop) of the global numbering that belong to group
// class k (G = 2^(k+1) lanes per cell) and fall to wavefront gwave.
// Items of 2..8-lane groups are short chains of dependent loads and a few
// steps of work, and a wavefront takes several per frame before the
// collapse: their loads are pipelined, the next item's cells and particles
// in flight while the current one computes.
template <int G>
__device__ __forceinline__ void group_class(const FrameParams &p, const FrameBuffers &b,
                                            const ItemMap &m, int k, uint32_t start,
                                            uint32_t stop, uint32_t gwave, uint32_t nwaves) {
    uint32_t v = gwave;
    if (v < start) v += (start - v + nwaves - 1) / nwaves * nwaves;
    if (v >= stop) return;
    uint32_t avail;
    const uint4 *list = locate(b, m, k, v - start, avail);
    if (G > 8) {
        for (;;) {
            group_run<G>(p, b, group_load<G>(b, group_entry<G>(list, avail)));
            v += nwaves;
            if (v >= stop) break;
            list = locate(b, m, k, v - start, avail);
        }
        return;
    }
    // Entries run two items ahead, particles one.
    GroupItem cur = group_load<G>(b, group_entry<G>(list, avail));
    uint4 ent = make_uint4(0, 0, 0, 0);
    if (v + nwaves < stop) {
        list = locate(b, m, k, v + nwaves - start, avail);
        ent = group_entry<G>(list, avail);
    }
    for (;;) {
        const uint32_t vn = v + nwaves;
        const bool more = vn < stop;
        GroupItem nxt;
        if (more) nxt = group_load<G>(b, ent);
        if (vn + nwaves < stop) {
            list = locate(b, m, k, vn + nwaves - start, avail);
            ent = group_entry<G>(list, avail);
        }
        group_run<G>(p, b, cur);
        if (!more) break;
        cur = nxt;
        v = vn;
    }
}

// Every queued cell:
//  1. class 6 (65..kWideMax particles), three cells per block item, on the
//     first blocks;
//  2. the group classes from 64 lanes per cell down to 2, wavefront work
//     items spread over every wavefront, numbered from the first block
//     without a class-6 item so that those take group work first;
//  3. class 7 (over kWideMax particles), one block each (block-wide LDS sort,
//     or merge sort past kLdsSort).
__global__ __launch_bounds__(kCollideBlock) void cells_kernel(FrameParams p, FrameBuffers b) {
    __shared__ union {
        struct {
            WaveLds w[kWavesPerBlock];
            WideStage stage;
        } wide;
        unsigned long long sort[kLdsSort];
    } sh;
    __shared__ ItemMap map;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t gwave = blockIdx.x * kWavesPerBlock + wave;
    const uint32_t nwaves = gridDim.x * kWavesPerBlock;
    build_item_map(b, map);
    __syncthreads();

    const uint32_t items6 = map.items[kWaveClass];
    for (uint32_t it = blockIdx.x; it < items6; it += gridDim.x) {
        uint32_t avail;
        const uint4 *list = locate(b, map, kWaveClass, it, avail);
        wide_item(p, b, list, avail, sh.wide.w, sh.wide.stage);
    }

    // end[k]: one past the last work item of group class k, largest first.
    uint32_t end[kGroupClasses];
    {
        uint32_t at = 0;
#pragma unroll
        for (int k = kGroupClasses - 1; k >= 0; --k) {
            at += map.items[k];
            end[k] = at;
        }
    }
    const uint32_t busy = (items6 < gridDim.x ? items6 : gridDim.x) * kWavesPerBlock;
    const uint32_t rw = gwave >= busy ? gwave - busy : gwave + nwaves - busy;
    // One loop per group class keeps each variant's registers to itself.
    group_class<64>(p, b, map, 5, 0, end[5], rw, nwaves);
    group_class<32>(p, b, map, 4, end[5], end[4], rw, nwaves);
    group_class<16>(p, b, map, 3, end[4], end[3], rw, nwaves);
    group_class<8>(p, b, map, 2, end[3], end[2], rw, nwaves);
    group_class<4>(p, b, map, 1, end[2], end[1], rw, nwaves);
    group_class<2>(p, b, map, 0, end[1], end[0], rw, nwaves);

    const uint32_t nb = map.items[kBlockClass];
    if (nb == 0) return;
    __syncthreads();
    for (uint32_t e = blockIdx.x; e < nb; e += gridDim.x) {
        uint32_t avail;
        const uint4 cell = *locate(b, map, kBlockClass, e, avail);
        big_cell<true>(p, b, cell.x, cell.y, cell.z, sh.sort);
    }
}

// The readback's canonical order, no arithmetic: one packed particle per
// lane as in collide_kernel, each copied to (its cell's start + its rank by
// source index).  A cell inside the wavefront's 64 particles is ranked with
// shuffles, a particle of a cell that runs past them counts the smaller
// sources of its cell itself (n loads that its lanes share), and
// of a cell over kWideMax particles, where that count would cost more than
// sorting, the block that holds its first particle sorts it (at most one a
// block).  1M loose particles: 13 us; a thread per cell over the 2.1M cells
// took 25, and its queue of large cells and the offsets three launches more
// (15 us).  The collapsed lattice, 2,000 cells of 460: 62 us, and 73 with a
// block sorting each of them from the queue.
//
// The blocks after the particles' fill the offsets: to b.idx those of the
// chunks the last scan found empty, or to `idx_out` all of them (no chunk is
// relative then: launch_canonical).
__global__ __launch_bounds__(kCollideBlock) void canonical_kernel(FrameParams p, FrameBuffers b,
                                                                  uint32_t *idx_out) {
    __shared__ unsigned long long sk[kLdsSort];
    __shared__ uint2 s_big;
    const uint32_t blocks = (p.n + kCollideBlock - 1) / kCollideBlock;
    if (*b.error) {  // raised before this kernel, if at all: no offsets are read, none are written
        if (!b.error_seen) return;
        const uint32_t i = blockIdx.x * kCollideBlock + threadIdx.x;
        if (b.keep_dead && i < p.n) {
            b.pos_out[i] = b.pos[i];
            b.vel_out[i] = b.vel[i];
        }
        __syncthreads();
        if (threadIdx.x == 0 && atomicAdd(b.error_seen, 1u) == gridDim.x - 1) {
            *b.error_seen = 0;
            *b.error = 0;
        }
        return;
    }
    if (blockIdx.x >= blocks) {
        const uint32_t chunk = blockIdx.x - blocks;
        const bool live = b.chunk_live[chunk] != 0;
        if (idx_out && chunk == 0 && threadIdx.x == 0) {
            idx_out[0] = 0;
            idx_out[p.ncell + 1] = p.n;
        }
        if (live && !idx_out) return;
        uint32_t *out = idx_out ? idx_out : b.idx;
        const uint32_t v = b.chunk_prefix[chunk];
#pragma unroll
        for (uint32_t i = 0; i < kChunkCells; i += kCollideBlock) {
            const uint32_t c = chunk * kChunkCells + i + threadIdx.x;
            if (c < p.ncell) out[1 + c] = live ? b.idx[1 + c] : v;
        }
        return;
    }
    if (threadIdx.x == 0) s_big = make_uint2(0, 0);
    __syncthreads();
    const uint32_t lane = lane_id();
    const uint32_t i0 = blockIdx.x * kCollideBlock + (threadIdx.x & ~63u), i = i0 + lane;
    const bool valid = i < p.n;
    const uint32_t k = valid ? b.key[i] : kNoKey;
    uint32_t before = kNoKey, after = kNoKey;
    if (lane == 0 && i0 > 0 && i0 < p.n) before = b.key[i0 - 1];
    if (lane == 63 && i0 + 64 < p.n) after = b.key[i0 + 64];
    uint32_t sv = 0;
    float2 q = make_float2(0.0f, 0.0f), w = q;
    if (valid) {
        sv = b.src[i] & kSrcMask;
        q = b.pos[i];
        w = b.vel[i];
    }
    const uint32_t kp = from_lane_before(k, before), kn = from_lane_after(k, after);
    const unsigned long long lt = lanemask_lt(), le = lt | (1ull << lane);
    const unsigned long long heads = __ballot(valid && k != kp), tails = __ballot(valid && k != kn);
    const unsigned long long hb = heads & le, ta = tails & ~lt;
    const int hl = hb ? 63 - (int)__builtin_clzll(hb) : -1;
    const int tl = ta ? (int)__builtin_ctzll(ta) : 64;
    const bool known = valid && k < p.ncell;  // a key past the grid: no layout writes one
    const bool inside = known && hl >= 0 && tl < 64;
    const uint32_t m = inside ? (uint32_t)(tl - hl + 1) : 0u;
    uint32_t rank = 0, s = inside ? i0 + (uint32_t)hl : 0u;
    bool write = inside;
    // Source indices inside a cell are distinct.
    const uint32_t mw = wave_max_u32(m);
    if (mw > 1)
        for (uint32_t t = 0; t < mw; ++t) {
            const bool in = t < m;
            const uint32_t o = (uint32_t)__shfl((int)sv, in ? hl + (int)t : (int)lane, 64);
            rank += (in && o < sv) ? 1u : 0u;
        }
    if (known && !inside) {
        uint32_t e;
        cell_range(p, b, k, s, e);
        const uint32_t n = e > s ? e - s : 0u;
        if (n > kWideMax) {
            if (i == s) s_big = make_uint2(s, n);
        } else {
            write = true;
            const uint32_t *src = b.src + s;
            uint32_t t = 0;
            for (; t + 16 <= n; t += 16) {
                uint32_t v[16];
#pragma unroll
                for (int u = 0; u < 16; ++u) v[u] = src[t + u];
#pragma unroll
                for (int u = 0; u < 16; ++u) rank += (v[u] & kSrcMask) < sv ? 1u : 0u;
            }
            for (; t + 4 <= n; t += 4)
#pragma unroll
                for (int u = 0; u < 4; ++u) rank += (src[t + u] & kSrcMask) < sv ? 1u : 0u;
            for (; t < n; ++t) rank += (src[t] & kSrcMask) < sv ? 1u : 0u;
        }
    }
    if (write && s + rank < p.n) {  // always within, with offsets that agree with the keys
        b.pos_out[s + rank] = q;
        b.vel_out[s + rank] = w;
    }
    __syncthreads();
    const uint2 big = s_big;
    if (big.y) big_cell<false>(p, b, big.x, big.y, 0, sk);
}

// ---------------------------------------------------------------------------
// Exclusive scan of the counts: one tile of THREADS x ITEMS cells per block; status
// words are tagged with the frame's epoch so they never need clearing.

constexpr unsigned long long kFlagAggregate = 1ull;
constexpr unsigned long long kFlagInclusive = 2ull;
constexpr uint32_t kEpochMask = 0x3fffffffu;
constexpr int kLookWindows = 4;  // 64-tile windows read per look-back round

__device__ __forceinline__ unsigned long long status_word(unsigned long long flag, uint32_t epoch,
                                                          uint32_t value) {
    return (flag << 62) | ((unsigned long long)(epoch & kEpochMask) << 32) | value;
}

// Exclusive prefix of `tile` from its predecessors' status words, by one
// wavefront.  Lane l of window w reads tile j - 64w - l.  A tile waits only
// on tiles dispatched before it, so the wait ends; should it not within
// p.wait_limit rounds, the tile raises kErrLookBack and takes 0 (the frame
// kernels clamp every offset range to the particles, so what follows stays
// in bounds, and the host reports the error).
__device__ uint32_t look_back(const FrameParams &p, const FrameBuffers &b, uint32_t tile,
                              uint32_t epoch) {
    const uint32_t lane = lane_id();
    uint32_t excl = 0;
    int64_t j = (int64_t)tile - 1;
    epoch = (epoch + p.epoch_skew) & kEpochMask;
    for (uint32_t round = 0;; ++round) {
        if (round >= p.wait_limit) {
            if (lane == 0) raise_error(b, kErrLookBack);
            return 0u;
        }
        unsigned long long w[kLookWindows];
#pragma unroll
        for (int q = 0; q < kLookWindows; ++q) {
            const int64_t jj = j - 64 * q - (int64_t)lane;
            w[q] = jj >= 0 ? __hip_atomic_load(&b.tile_state[jj], __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT)
                           : status_word(kFlagInclusive, epoch, 0);
        }
        bool finished = false, stalled = false;
#pragma unroll
        for (int q = 0; q < kLookWindows; ++q) {
            if (!finished && !stalled) {
                const unsigned long long flag = w[q] >> 62;
                const bool ok = flag != 0 && (uint32_t)((w[q] >> 32) & kEpochMask) == epoch;
                const unsigned long long okm = __ballot(ok);
                const unsigned long long incm = __ballot(ok && flag == kFlagInclusive);
                const uint32_t val = (uint32_t)w[q];
                if (incm != 0) {
                    const int first = __builtin_ctzll(incm);
                    const unsigned long long need =
                        first == 63 ? ~0ull : ((1ull << (first + 1)) - 1);
                    if ((okm & need) == need) {
                        excl += wave_sum((int)lane <= first ? val : 0u);
                        finished = true;
                    } else {
                        stalled = true;
                    }
                } else if (okm == ~0ull) {
                    excl += wave_sum(val);
                    j -= 64;
                } else {
                    stalled = true;
                }
            }
        }
        if (finished) return excl;
        if (stalled) __builtin_amdgcn_s_sleep(1);
    }
}

// By the first wavefront of a tile with total `agg`: publishes it, finds the
// tile's exclusive prefix and publishes that.
__device__ __forceinline__ uint32_t publish_tile(const FrameParams &p, const FrameBuffers &b, uint32_t tile,
                                                 uint32_t epoch, uint32_t agg) {
    const uint32_t lane = lane_id();
    uint32_t excl = 0;
    if (tile == 0) {
        if (lane == 0)
            __hip_atomic_store(&b.tile_state[0], status_word(kFlagInclusive, epoch, agg), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    } else {
        if (lane == 0)
            __hip_atomic_store(&b.tile_state[tile], status_word(kFlagAggregate, epoch, agg), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        excl = look_back(p, b, tile, epoch);
        if (lane == 0)
            __hip_atomic_store(&b.tile_state[tile], status_word(kFlagInclusive, epoch, excl + agg), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
    return excl;
}

// THREADS x ITEMS counts per tile (kScanShapes); ITEMS is a multiple of 4.
template <int THREADS, int ITEMS>
__global__ __launch_bounds__(THREADS) void scan_kernel(FrameParams p, FrameBuffers b) {
    static_assert(ITEMS % 4 == 0 && THREADS % 64 == 0, "128-bit count loads, whole wavefronts");
    __shared__ uint32_t s_prefix;
    __shared__ uint32_t s_wave[THREADS / 64];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63, wave = tid >> 6;
    // Tiles follow block order: a block waits only on lower-numbered blocks,
    // which were dispatched before it.
    const uint32_t tile = blockIdx.x;
    const uint32_t epoch = *b.epoch & kEpochMask;
    const uint32_t base = tile * (THREADS * ITEMS) + tid * ITEMS;
    // A chunk in which no slot was claimed this frame holds only zero counts:
    // its counts are not read and its offsets not written (the readback fills
    // them in from chunk_prefix).
    const uint32_t chunk = base >> kChunkShift;
    const bool live = base < p.ncell && b.chunk_next[chunk] != 0;

    // Load ITEMS counts and clear them for the next frame.
    uint32_t v[ITEMS];
    if (!live) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) v[i] = 0;
    } else if (base + ITEMS <= p.ncell) {
        uint4 *q = reinterpret_cast<uint4 *>(b.cnt + base);
#pragma unroll
        for (int i = 0; i < ITEMS / 4; ++i) {
            const uint4 w = q[i];
            v[4 * i] = w.x; v[4 * i + 1] = w.y; v[4 * i + 2] = w.z; v[4 * i + 3] = w.w;
        }
        // Clear only what holds counts: after the first frames most of the
        // grid is empty, and these stores are a third of the kernel's bytes.
#pragma unroll
        for (int i = 0; i < ITEMS / 4; ++i)
            if (v[4 * i] | v[4 * i + 1] | v[4 * i + 2] | v[4 * i + 3]) q[i] = make_uint4(0, 0, 0, 0);
    } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (base + i < p.ncell) {
                v[i] = b.cnt[base + i];
                b.cnt[base + i] = 0;
            } else {
                v[i] = 0;
            }
        }
    }
    uint32_t mine = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) mine += v[i];
    const uint32_t incl = wave_inclusive_sum(mine);
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    uint32_t wave_off = 0, agg = 0;
#pragma unroll
    for (int w = 0; w < THREADS / 64; ++w) {
        const uint32_t ws = s_wave[w];
        if ((uint32_t)w < wave) wave_off += ws;
        agg += ws;
    }

    if (wave == 0) {
        const uint32_t excl = publish_tile(p, b, tile, epoch, agg);
        if (lane == 0) s_prefix = excl;
    }
    __syncthreads();

    // idx[1 + k] = start_k; idx[0] = 0; idx[C + 1] = N.
    uint32_t run = s_prefix + wave_off + incl - mine;
    uint32_t out[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        out[i] = run;
        run += v[i];
    }
    uint32_t *dst = b.idx + 1 + base;
    if (!live) {
    } else if (base + ITEMS <= p.ncell) {
        uint4 *q = reinterpret_cast<uint4 *>(dst);
#pragma unroll
        for (int i = 0; i < ITEMS / 4; ++i)
            q[i] = make_uint4(out[4 * i], out[4 * i + 1], out[4 * i + 2], out[4 * i + 3]);
    } else {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            if (base + i < p.ncell) dst[i] = out[i];
    }
    if ((base & (kChunkCells - 1)) == 0 && base < p.ncell) {  // the chunk's first thread
        b.chunk_prefix[chunk] = out[0];
        b.chunk_live[chunk] = live ? kChunkWhole : kChunkEmpty;
        b.chunk_next[chunk] = 0;  // every thread of the chunk read it before the barriers above
    }
    if (tile == 0 && tid == 0) {
        b.idx[0] = 0;
    }
    if (tile == 0)  // the cell kernel of this frame has finished with the lists
        for (uint32_t i = tid; i < (uint32_t)(kClasses * (kSlices + 1)); i += THREADS)
            b.class_ctr[i * kCtrStride] = 0;
    if (tile == b.scan_tiles - 1 && tid == 0) b.idx[p.ncell + 1] = s_prefix + agg;
}

// The scan of large grids (relative_offsets), in two launches without a wait
// between tiles of cells: every live chunk scanned by itself by one
// wavefront, its offsets left counted from its own first cell, and then the
// chunks' totals scanned (chunk_scan_kernel), which makes the chunks' first
// offsets.  Readers add the two.  Counted so they fit 16 bits, which halves
// what this kernel writes and what the scatter gathers; a chunk of more
// particles than that has kWideOffset there and its offsets in idx.  The
// counts are read and cleared past the caches (nontemporal): the offsets,
// which the scatter reads next, stay in them.
//
// One pass over the cells (scan_kernel) holds its counts in registers until
// its look-back ends, two tiles of 32k cells on a CU, one loading while the
// other waits.  512 worlds of 227M cells, half the chunks live: 345 us in one
// pass, 107 + 6 here (0.45 GB of counts read and 0.23 GB written), and with
// 32-bit offsets 137 + 6.  4M particles on 16.8M cells: 49 us, 23 + 6 here,
// and their scatter 54 and 45 (53 with the counts read through the caches).
// The 2.1M cells of the 1M lattice take 7.4 us in one pass, hardly more than
// two launches cost; hence the line at 2^23 cells, where the pass needed
// larger tiles already.
//
// A wavefront looks after `per` consecutive chunks: as few as leave every
// wavefront slot of the device one (kChipWaves), at most kWaveChunks (4, 16:
// 144 and 168 us instead of 137 on the 227M cells: the chunks in flight lie
// farther apart).
constexpr uint32_t kWaveChunks = 2, kChipWaves = 8192;

__device__ __forceinline__ uint4 load_past(const uint4 *p) {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    const u4 v = __builtin_nontemporal_load(reinterpret_cast<const u4 *>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ void clear_past(uint4 *p) {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    const u4 zero = {0, 0, 0, 0};
    __builtin_nontemporal_store(zero, reinterpret_cast<u4 *>(p));
}

__global__ __launch_bounds__(256) void cell_scan_kernel(FrameParams p, FrameBuffers b, uint32_t chunks, uint32_t per) {
    const uint32_t lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t c0 = (blockIdx.x * 4 + wave) * per;
    // The cell kernel of this frame has finished with the lists.
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < (uint32_t)(kClasses * (kSlices + 1)); i += gridDim.x * 256)
        b.class_ctr[i * kCtrStride] = 0;
    if (c0 >= chunks) return;
    const bool mine = lane < per && c0 + lane < chunks;
    const uint32_t marked = mine ? b.chunk_next[c0 + lane] : 0u;
    uint32_t total = 0;  // lane l: of chunk c0 + l
    for (unsigned long long left = __ballot(marked != 0); left; left &= left - 1) {
        const uint32_t which = (uint32_t)__builtin_ctzll(left), c = c0 + which;
        const uint32_t base = c * kChunkCells + 4 * lane;  // cells base + 256u .. + 3
        uint4 v[4], at[4];
        if (c * kChunkCells + kChunkCells <= p.ncell) {
            uint4 *q = reinterpret_cast<uint4 *>(b.cnt + base);
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = load_past(q + 64 * u);
            // Clear only what holds counts: most cells of a large grid are empty.
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (v[u].x | v[u].y | v[u].z | v[u].w) clear_past(q + 64 * u);
        } else {  // the grid's last chunk
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                uint32_t w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t k = base + 256 * u + e;
                    w[e] = k < p.ncell ? b.cnt[k] : 0u;
                    if (k < p.ncell) b.cnt[k] = 0;
                }
                v[u] = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
        uint32_t run = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t sum = v[u].x + v[u].y + v[u].z + v[u].w;
            const uint32_t incl = wave_inclusive_sum(sum);
            at[u].x = run + incl - sum;
            at[u].y = at[u].x + v[u].x;
            at[u].z = at[u].y + v[u].y;
            at[u].w = at[u].z + v[u].z;
            run += __builtin_amdgcn_readlane(incl, 63);
        }
        uint2 *rel = reinterpret_cast<uint2 *>(b.rel + base);  // whole chunks long
        const bool wide = run >= kWideOffset;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            rel[64 * u] = wide ? make_uint2(~0u, ~0u)
                               : make_uint2(at[u].x | at[u].y << 16, at[u].z | at[u].w << 16);
        if (wide || p.idx_read) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t w[4] = {at[u].x, at[u].y, at[u].z, at[u].w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (base + 256 * u + e < p.ncell) b.idx[1 + base + 256 * u + e] = w[e];
            }
        }
        total = lane == which ? run : total;
    }
    if (mine) {
        b.chunk_sum[c0 + lane] = total;
        b.chunk_live[c0 + lane] = marked ? kChunkRelative : kChunkEmpty;
        b.chunk_next[c0 + lane] = 0;
    }
}

// Exclusive scan of the chunks' totals into chunk_prefix: the single-pass
// scan of scan_kernel, a tile of kChunkTile chunks a block.
__global__ __launch_bounds__(1024) void chunk_scan_kernel(FrameParams p, FrameBuffers b, uint32_t chunks) {
    constexpr uint32_t kItems = kChunkTile / 1024;
    __shared__ uint32_t s_prefix;
    __shared__ uint32_t s_wave[16];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t tile = blockIdx.x;
    const uint32_t epoch = *b.epoch & kEpochMask;
    const uint32_t base = tile * kChunkTile + threadIdx.x * kItems;
    uint32_t v[kItems], mine = 0;
#pragma unroll
    for (uint32_t i = 0; i < kItems; ++i) {
        v[i] = base + i < chunks ? b.chunk_sum[base + i] : 0u;
        mine += v[i];
    }
    const uint32_t incl = wave_inclusive_sum(mine);
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    uint32_t wave_off = 0, agg = 0;
#pragma unroll
    for (uint32_t w = 0; w < 16; ++w) {
        const uint32_t ws = s_wave[w];
        if (w < wave) wave_off += ws;
        agg += ws;
    }
    if (wave == 0) {
        const uint32_t excl = publish_tile(p, b, tile, epoch, agg);
        if (lane == 0) s_prefix = excl;
    }
    __syncthreads();
    uint32_t run = s_prefix + wave_off + incl - mine;
#pragma unroll
    for (uint32_t i = 0; i < kItems; ++i) {
        if (base + i < chunks) b.chunk_prefix[base + i] = run;
        run += v[i];
    }
    if (tile == 0 && threadIdx.x == 0) b.idx[0] = 0;
    if (tile == gridDim.x - 1 && threadIdx.x == 0) b.idx[p.ncell + 1] = s_prefix + agg;
}

// ---------------------------------------------------------------------------

// PER particles per lane (kScatterPerLane), strided across the wavefront: every
// load of the dependent chain (kslot -> start offset -> destination) is in
// flight for all of them at once.
// RELATIVE: the offsets are 16 bits from their chunk's prefix
// (relative_offsets).  A template: with the choice made at run time 4M loose
// particles took 57 us instead of 45 (whole offsets: 54), and the 1M lattice
// 12.5 instead of 11.8 where one form of loads serves both.
template <int PER, bool RELATIVE>
__global__ __launch_bounds__(kScatterBlock) void scatter_kernel(FrameParams p, FrameBuffers b) {
    // Blocks go to the 8 XCDs in turn (block b to XCD b % 8): block b takes
    // tile (b % 8) * (grid / 8) + b / 8, so that each XCD scatters one
    // contiguous eighth of the particles.  Their destinations then share
    // lines mostly with destinations of the same XCD, whose L2 merges the
    // partial lines before writing them back.  The grid is a multiple of 8.
    const uint32_t tile = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const uint32_t w0 = (tile * kScatterBlock + (threadIdx.x & ~63u)) * PER;
    const uint32_t ln = threadIdx.x & 63;
    if (blockIdx.x == 0 && threadIdx.x == 0) *b.epoch = *b.epoch + 1;  // the frame's scan has finished
    uint2 ks[PER];
    float2 q[PER], v[PER];
    uint32_t start[PER], prefix[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const uint32_t i = w0 + 64 * j + ln;
        if (i < p.n) {
            ks[j] = b.kslot[i];
            q[j] = b.pos_out[i];
            v[j] = b.vel_out[i];
        }
    }
    // A scan that gave up its look-back (b.error) left offsets that are not
    // valid: the scatter then writes nothing (a vector load beside the
    // others, checked before the stores).
    const uint32_t dead = b.error[lane_id() >> 6];
#pragma unroll
    for (int j = 0; j < PER; ++j)
        if (w0 + 64 * j + ln < p.n) {
            if (RELATIVE) {
                start[j] = reinterpret_cast<const uint16_t *>(b.off)[ks[j].x];
                prefix[j] = b.chunk_prefix[ks[j].x >> kChunkShift];
            } else {
                start[j] = b.idx[ks[j].x + 1];
            }
        }
    if (__builtin_amdgcn_readfirstlane(dead)) return;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const uint32_t i = w0 + 64 * j + ln;
        if (i < p.n) {
            uint32_t dest = start[j] + (ks[j].y & kSrcMask);
            if (RELATIVE) {
                if (start[j] == kWideOffset) dest = b.idx[ks[j].x + 1] + (ks[j].y & kSrcMask);
                dest += prefix[j];
            }
            if (dest < p.n) {  // always, with a consistent frame
                b.pos[dest] = q[j];
                b.vel[dest] = v[j];
                b.src[dest] = i | (ks[j].y & kRunFlag);
                b.key[dest] = ks[j].x;
            }
        }
    }
}

// Whole offsets in idx everywhere: an empty chunk's entries become the offset
// at its first cell, a relative chunk's theirs counted from 0, and it is whole
// then.
__global__ __launch_bounds__(256) void materialize_kernel(FrameParams p, FrameBuffers b) {
    const uint32_t chunk = blockIdx.x;
    const uint32_t state = b.chunk_live[chunk];
    if (state == kChunkWhole) return;
    const uint32_t v = b.chunk_prefix[chunk];
    for (uint32_t i = threadIdx.x; i < kChunkCells; i += 256) {
        const uint32_t c = chunk * kChunkCells + i;
        uint32_t at = 0;
        if (c < p.ncell && state == kChunkRelative) {
            at = offset_entry(b, c, offset_word(b, c));
            if (at == kWideOffset) at = b.idx[1 + c];
        }
        if (c < p.ncell) b.idx[1 + c] = v + at;
    }
    __syncthreads();  // every thread has read the state
    if (threadIdx.x == 0 && state == kChunkRelative) b.chunk_live[chunk] = kChunkWhole;
}

__global__ void copy32_kernel(uint32_t *dst, const uint32_t *src, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

__global__ void iota_kernel(uint32_t *dst, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = i;
}

// key[i]: the last cell c whose start idx[c + 1] is at most i (offsets given
// whole, non-decreasing from idx[1] = 0, so that cell's range holds i).
__global__ void keys_from_offsets_kernel(const uint32_t *idx, uint32_t ncell, uint32_t n,
                                         uint32_t *key) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t lo = 0, hi = ncell;  // idx[lo + 1] <= i < idx[hi + 1] (idx[ncell + 1] = n)
    while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (idx[mid + 1] <= i) lo = mid;
        else hi = mid;
    }
    key[i] = lo;
}

// What a frame on a caller's packed triple starts from (wrach_frame_noalloc):
// the buffers that a context keeps clean between frames, cleared, and each
// particle's source index and cell from the caller's offsets.  One thread
// per cell, a cell of more than kOwnCells particles by its whole wavefront.
// Offsets that do not ascend from 0 to n are an error: the kernels that follow
// do nothing and the caller's arrays stay as they are.  (b.error is clear: the
// canonical kernel clears what a call raised.)  Such ranges may overlap, so
// one of more than kLongCell particles looks now and then whether another
// thread has found them wrong.
// One launch in place of 12 (nine fills, a copy, an iota and a binary search
// per particle), each 1.3 to 7 us and 2.7 us of the host's time.
__global__ __launch_bounds__(256) void noalloc_init_kernel(FrameParams p, FrameBuffers b,
                                                           const uint32_t *indices, uint32_t tiles,
                                                           uint32_t chunks) {
    constexpr uint32_t kOwnCells = 8, kLongCell = 1024;
    const uint32_t t = blockIdx.x * 256 + threadIdx.x, all = gridDim.x * 256;
    uint32_t s = 0, e = 0;
    bool bad = false;
    if (t < p.ncell) {  // the grid covers the cells
        s = indices[1 + t];
        e = indices[2 + t];
        bad = e < s || e > p.n || (t == 0 && s != 0) || (t == p.ncell - 1 && e != p.n);
    }
    const unsigned long long any = __ballot(bad);
    if (any && lane_id() == (uint32_t)__builtin_ctzll(any)) raise_error(b, kErrLayout);
    const uint32_t n = bad ? 0u : e - s;
    for (uint32_t i = t; i < p.ncell + 16; i += all) b.cnt[i] = 0;
    for (uint32_t i = t; i < tiles; i += all) b.tile_state[i] = 0;
    for (uint32_t i = t; i < chunks; i += all) {
        b.chunk_next[i] = 0;
        b.chunk_live[i] = 1;  // every offset is the caller's
    }
    for (uint32_t i = t; i < (uint32_t)(kClasses * (kSlices + 1)); i += all) b.class_ctr[i * kCtrStride] = 0;
    if (t == 0) {
        *b.epoch = 1;  // status words start at 0, never valid
    }
    if (n <= kOwnCells)
        for (uint32_t j = s; j < s + n; ++j) {
            b.src[j] = j;
            b.key[j] = t;
        }
    unsigned long long big = __ballot(n > kOwnCells);
    while (big) {
        const int l = __builtin_ctzll(big);
        big &= big - 1;
        const uint32_t s0 = (uint32_t)__shfl((int)s, l, 64), n0 = (uint32_t)__shfl((int)n, l, 64);
        const uint32_t c0 = (uint32_t)__shfl((int)t, l, 64);
        for (uint32_t r = 0; r < n0; r += kLongCell) {
            if (r && __hip_atomic_load(b.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
            for (uint32_t j = s0 + r + lane_id(); j < s0 + min(n0, r + kLongCell); j += 64) {
                b.src[j] = j;
                b.key[j] = c0;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Upload binning (SpatialBin::create_packed_data, spatial_bin.rs:103-149, on
// the device).  The CPU packer is a stable counting sort of the store by
// cell; here each particle takes a slot with one atomic, so a cell's
// particles land in arbitrary order, each marked as a run of its own.  The
// order inside a cell is then the one every frame already restores (runs
// ordered by source index, here the store index), and the readback's
// canonical pass applies it as well: the packed triple is the CPU packer's.

// Rust's `f as i32`: saturating, NaN -> 0.
__device__ __forceinline__ int32_t saturating_i32(float f) {
    if (f != f) return 0;
    if (f >= 2147483648.0f) return 0x7fffffff;
    if (f <= -2147483648.0f) return (int32_t)0x80000000u;
    return (int32_t)f;
}

// f32::div_euclid for b > 0 (spatial_bin.rs:48-64): the truncated IEEE
// quotient, one less when the remainder is negative.
__device__ __forceinline__ float div_euclid_pos(float a, float b) {
    const float q = truncf(a / b);
    return fmodf(a, b) < 0.0f ? q - 1.0f : q;
}

// The packer's cell of a store particle (spatial_bin.rs:48-64) in a grid of
// gx x gy cells; false outside it.
__device__ __forceinline__ bool store_cell(const UploadParams &u, float2 q, uint32_t gx, uint32_t gy,
                                           uint32_t &key) {
    // The cell relative to the grid's bottom-left cell (the view anchor's).
    const int64_t cx = (int64_t)saturating_i32(div_euclid_pos(q.x, u.cs)) - u.blx;
    const int64_t cy = (int64_t)saturating_i32(div_euclid_pos(q.y, u.cs)) - u.bly;
    const bool in = cx >= 0 && cy >= 0 && cx < (int64_t)gx && cy < (int64_t)gy;
    key = in ? (uint32_t)cy * gx + (uint32_t)cx : 0xffffffffu;
    return in;
}

__global__ __launch_bounds__(256) void upload_bin_kernel(UploadParams u, FrameBuffers b) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    bool in = false;
    if (i < u.n) {
        uint2 ks = make_uint2(0xffffffffu, 0u);
        // Its world's grid in a batch: worlds of one size one after another,
        // or each world's own grid.
        uint32_t gx = u.gx, gy = u.gy, base = 0;
        if (u.world) {
            if (u.grids) {
                const WorldGrid g = u.grids[u.world[i]];
                gx = g.gx;
                gy = g.gy;
                base = g.base;
            } else {
                base = u.world[i] * u.world_cells;
            }
        }
        in = store_cell(u, u.pos[i], gx, gy, ks.x);
        if (in) {
            ks.x += base;
            ks.y = claim(b, ks.x, 1u);
        }
        u.ks[i] = ks;
    }
    // Outside the grid, striped: a wavefront's atomic for the particles inside
    // serialised on one counter (184 us for 1M particles, 12 ns a wavefront).
    const unsigned long long m = __ballot(i < u.n && !in);
    if (lane_id() == 0 && m != 0)
        atomicAdd(&u.outside[(blockIdx.x % kOutsideStripes) * kCtrStride], (uint32_t)__popcll(m));
}

// The striped counts' sum, to host memory (a copy of the counters would be
// the upload's only one to the host).
__global__ __launch_bounds__(64) void outside_sum_kernel(const uint32_t *outside, uint32_t *host) {
    static_assert(kOutsideStripes <= 64, "a counter per lane");
    const uint32_t t = threadIdx.x;
    const uint32_t sum = wave_sum(t < kOutsideStripes ? outside[t * kCtrStride] : 0u);
    if (t == 0) __hip_atomic_store(host, sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The store's particles outside the grid, appended at dpos/dvel[base + ...]
// (wrach_store_write_back) in their store order: a moved view can bring
// them into cells later, where that order is their in-cell order.  Two
// launches: each block counts its own (counts[block]); the host turns the
// counts into exclusive offsets; each block then writes its particles from
// its offset on, ranked within the block by ballots.
__global__ __launch_bounds__(256) void store_outside_count_kernel(UploadParams u, uint32_t *counts) {
    __shared__ uint32_t s_n[4];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    bool out = false;
    if (i < u.n) {
        uint32_t key;
        out = !store_cell(u, u.pos[i], u.gx, u.gy, key);
    }
    const unsigned long long m = __ballot(out);
    if (lane_id() == 0) s_n[threadIdx.x >> 6] = (uint32_t)__popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = s_n[0] + s_n[1] + s_n[2] + s_n[3];
}

__global__ __launch_bounds__(256) void store_outside_kernel(UploadParams u, float2 *dpos,
                                                            float2 *dvel, uint32_t base,
                                                            const uint32_t *offsets) {
    __shared__ uint32_t s_n[4];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    bool out = false;
    float2 q = make_float2(0.0f, 0.0f);
    if (i < u.n) {
        q = u.pos[i];
        uint32_t key;
        out = !store_cell(u, q, u.gx, u.gy, key);
    }
    const unsigned long long m = __ballot(out);
    const uint32_t wave = threadIdx.x >> 6;
    if (lane_id() == 0) s_n[wave] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < wave; ++w) before += s_n[w];
    if (out) {
        const uint32_t j = base + offsets[blockIdx.x] + before + (uint32_t)__popcll(m & lanemask_lt());
        dpos[j] = q;
        dvel[j] = u.vel[i];
    }
}

__global__ __launch_bounds__(256) void upload_scatter_kernel(UploadParams u, FrameBuffers b) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x == 0) *b.epoch = *b.epoch + 1;  // the scan has finished
    if (i >= u.n) return;
    const uint2 ks = u.ks[i];
    if (ks.x == 0xffffffffu) return;
    uint32_t at = offset_entry(b, ks.x, offset_word(b, ks.x));  // the chunk is live
    if (b.off_shift) at = wide_entry(b, ks.x, at, kChunkRelative) + b.chunk_prefix[ks.x >> kChunkShift];
    const uint32_t dest = at + ks.y;
    if (dest >= u.cap) return;  // never, with a consistent scan
    b.pos[dest] = u.pos[i];
    b.vel[dest] = u.vel[i];
    b.src[dest] = i | kRunFlag;
    b.key[dest] = ks.x;
}

// ---------------------------------------------------------------------------
// Mode S: separation passes over the 3x3 cells around each particle, before
// the reference step (an extension: the reference collides within one cell,
// shaders/physics/src/cell.rs:60-69).  A pass is Jacobi -- every particle
// reads the positions the pass started from -- and a particle's pair terms
// are rounded to multiples of 2^-30 and summed exactly, so its
// displacement does not depend on the order of the particles inside a cell
// (which the device layout keeps canonical only through `src`).

// A term is below 0.62 in magnitude (|dx| / d is at most 1 + 2^-22, or
// 1.22 where dx * dx is subnormal), so term * 2^30 is below 2^31 and
// rintf (round half to even, as llrintf) makes it an integer-valued float.
// The terms are summed as doubles: integers below 2^53 add exactly, and at
// most kStencilBudget of them stay far below that, so the double holds the
// same integer as an int64 sum, in two instructions a term in place of
// five (conversion, sign extension, 64-bit add).
constexpr float kStencilScale = 1073741824.0f;            // 2^30
constexpr float kStencilUnit = 9.313225746154785e-10f;    // 2^-30

// sqrtf(x) for x in [2^-96, 1 + 2^-23]: the hardware reciprocal root y,
// s = x * y, and one Newton step on the residual, fma(x - s * s, y / 2, s).
// That this equals the correctly rounded root for every x of the range is
// a property of the hardware reciprocal root, not a theorem;
// check_pair_arithmetic_kernel tests it for all 805,306,370 values of x on
// the device in use (wrach_check_pair_arithmetic).  hipcc's sqrtf takes
// v_sqrt_f32 (one unit in the last place either way), corrects it with
// two residual tests, and scales inputs below 2^-96.
__device__ __forceinline__ float sqrt_rn_above_2m96(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    const float s = x * y;
    const float e = __builtin_fmaf(-s, s, x);
    return __builtin_fmaf(e, 0.5f * y, s);
}

// (1 - d) * 2^29 / d correctly rounded, for d in [2^-48, 1] (so 1 - d is
// the overlap and the numerator a = (1 - d) * 2^29 is 0 or in
// [2^5, 2^29]): the hardware reciprocal y of d, the quotient a * y and one
// residual correction fma(fma(-d, q, a), y, q).  hipcc's f32 division adds
// a Newton step on y, a second correction, and v_div_scale / v_div_fixup
// (identities here: the exponent difference stays below 96, nothing is
// subnormal, and the fix-up only rewrites special operands).  That the
// short sequence equals the correctly rounded quotient for every d of the
// range is not a theorem but a property of the hardware reciprocal;
// check_pair_arithmetic_kernel tests it for all 402,653,185 values of d
// on the device in use (wrach_check_pair_arithmetic).
__device__ __forceinline__ float overlap_force_rn(float d) {
    const float a = (1.0f - d) * 0x1p29f;
    const float y = __builtin_amdgcn_rcpf(d);
    const float q = a * y;
    const float r = __builtin_fmaf(-d, q, a);
    return __builtin_fmaf(r, y, q);
}


// The pair arithmetic's short sequences against hipcc's correctly rounded
// ones over their whole input ranges: sqrt_rn_above_2m96(x) against
// sqrtf(x) for every float x in [2^-96, 1 + 2^-23], overlap_force_rn(d)
// against ((1 - d) * 2^29) / d for every float d in [2^-48, 1].  Adds the
// mismatches to out[0] and out[1] and the inputs tried to out[2] and
// out[3] (one atomic per wavefront and counter).
__global__ __launch_bounds__(256) void check_pair_arithmetic_kernel(unsigned long long *out) {
    const uint32_t s_lo = __float_as_uint(0x1p-96f), s_hi = __float_as_uint(1.00000011920928955078125f);
    const uint32_t d_lo = __float_as_uint(0x1p-48f), d_hi = __float_as_uint(1.0f);
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t t0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t bad_s = 0, bad_d = 0, n_s = 0, n_d = 0;
    for (uint64_t u = s_lo + t0; u <= s_hi; u += stride) {
        const float x = __uint_as_float((uint32_t)u);
        bad_s += __float_as_uint(sqrt_rn_above_2m96(x)) != __float_as_uint(sqrtf(x));
        ++n_s;
    }
    for (uint64_t u = d_lo + t0; u <= d_hi; u += stride) {
        const float d = __uint_as_float((uint32_t)u);
        const float full = ((1.0f - d) * 0x1p29f) / d;
        bad_d += __float_as_uint(overlap_force_rn(d)) != __float_as_uint(full);
        ++n_d;
    }
    const uint32_t v[4] = {wave_sum(bad_s), wave_sum(bad_d), wave_sum(n_s), wave_sum(n_d)};
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 4; ++k)
            if (v[k]) atomicAdd(&out[k], (unsigned long long)v[k]);
}

// The particles of the 3x3 cells around (cx, cy) as three ranges, one per
// row cy - 1 .. cy + 1: the cells of one row are contiguous in the packed
// layout, and [start(x0), start(x1 + 1)) covers columns x0..x1 (past the
// row's last column, start(x1 + 1) is the next row's first cell, which
// begins where the row ends).  `own`: the start of cell (cx, cy) itself.
// Every load is issued before the first is used (cell_start as a branch on
// the chunk's flag made 12 dependent loads of the six offsets).
__device__ __forceinline__ void stencil_rows(const FrameParams &p, const FrameBuffers &b,
                                             const Grid &g, int cx, int cy, uint32_t rs[3],
                                             uint32_t re[3], uint32_t &own) {
    const int gx = (int)g.gx, gy = (int)g.gy;
    const int x0 = cx > 0 ? cx - 1 : 0, x1 = cx + 1 < gx ? cx + 1 : gx - 1;
    // Cells: [2t] the first of row t, [2t + 1] past its last, [6] the own one.
    uint32_t c[7], at[7], live[7], pre[7];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        int y = cy + t - 1;
        y = y < 0 ? 0 : y < gy ? y : gy - 1;  // a row outside the world: loaded, not used
        c[2 * t] = g.base + (uint32_t)(y * gx + x0);
        c[2 * t + 1] = g.base + (uint32_t)(y * gx + x1 + 1);
    }
    c[6] = g.base + (uint32_t)(cy * gx + cx);
#pragma unroll
    for (int u = 0; u < 7; ++u) {
        const uint32_t k = c[u] < p.ncell ? c[u] : p.ncell - 1;
        live[u] = b.chunk_live[k >> kChunkShift];
        pre[u] = b.chunk_prefix[k >> kChunkShift];
        at[u] = b.idx[k + 1];  // also on large grids: FrameParams::idx_read
    }
#pragma unroll
    for (int u = 0; u < 7; ++u) {
        at[u] = offset_of(at[u], live[u], pre[u]);
        at[u] = c[u] < p.ncell && at[u] < p.n ? at[u] : p.n;
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        const int y = cy + t - 1;
        const bool in = y >= 0 && y < gy;  // the world's own rows only
        rs[t] = in ? at[2 * t] : 0u;
        re[t] = in && at[2 * t + 1] > at[2 * t] ? at[2 * t + 1] : rs[t];
    }
    own = at[6];
}

// The grid of the world that holds packed particle i: the last world whose
// first cell starts at or before i (an empty world starts where the next
// one does, so it is never the last such).  One world: its own grid.
__device__ __forceinline__ Grid particle_grid(const FrameParams &p, const FrameBuffers &b, uint32_t i) {
    if (p.grids) {
        uint32_t lo = 0, hi = p.n_grids;  // world lo starts at or before i
        while (hi - lo > 1) {
            const uint32_t mid = lo + (hi - lo) / 2;
            if (cell_start(p, b, p.grids[mid].base) <= i) lo = mid;
            else hi = mid;
        }
        return grid_of(p, p.grids[lo].base);
    }
    if (p.world_cells == p.ncell) return grid_of(p, 0u);
    uint32_t lo = 0, hi = p.ncell / p.world_cells;
    while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (cell_start(p, b, mid * p.world_cells) <= i) lo = mid;
        else hi = mid;
    }
    return grid_of(p, lo * p.world_cells);
}

// collide_pair's rule for particle i alone, given dx = x_i - x_j and
// dy = y_i - y_j: whether j is within reach, the overlap 1 - d (a multiple
// of 2^-24 in [0, 1]) and F = f * 2^30 for f = (0.5 * (1 - d)) / d.  The
// reference subtracts (p_j - p_i) * f from p_i (particles.rs:65-92), which
// is exactly (dx, dy) * f added: p_j - p_i = -(p_i - p_j) in IEEE
// arithmetic, up to the sign of a zero, which the rounding of the term to
// 2^-30 units drops.  That term, rint((dx * f) * 2^30), is rint(dx * F):
// f is 0 or at least 2^-25 (normal), so F is exactly f * 2^30, and
// dx * f * 2^30 rounds as dx * f does, scaled, unless dx * f is subnormal,
// where both round to 0.
constexpr float kReachSq = 1.00000011920928955078125f;  // 1 + 2^-23

// ov and F of a pair within reach at squared distance sq.
__device__ __forceinline__ void stencil_terms(float sq, float &ov, float &F) {
    if (sq < 0x1p-96f) {  // d below 2^-48, or 0: the full sequences
        float d = sqrtf(sq);
        if (d == 0.0f) d = 0.0001f;
        ov = 1.0f - d;
        F = ((0.5f * ov) / d) * kStencilScale;
        return;
    }
    const float d = sqrt_rn_above_2m96(sq);  // in [2^-48, 1]: never 0
    ov = 1.0f - d;
    // d is in [2^-48, 1]: overlap_force_rn's range, and the quotient is
    // (0.5 * ov / d) * 2^30 exactly, as f is normal.
    F = overlap_force_rn(d);
}

// `other`: j is not i (tested with the distance, so that the caller's load
// of p_j need not wait for it).
__device__ __forceinline__ bool stencil_reach(float dx, float dy, bool other, float &ov, float &F) {
    float sq = dx * dx;
    sq = sq + dy * dy;
    // sqrtf(sq) > 1 exactly when sq > 1 + 2^-23: sqrtf(1 + 2^-23) rounds to
    // 1 and the root of the next float above it does not, so d <= 1 below.
    // Most neighbours of a crowded cell are out of reach; they skip the root
    // and the division with the same outcome.
    if (!other | (sq > kReachSq)) return false;
    stencil_terms(sq, ov, F);
    return true;
}

// The sums of a particle's pairs.  ov is a multiple of 2^-24 in [0, 1], so
// a lane's sum of at most kStencilBudget of them is a multiple of 2^-24
// below 2^12: exact in a double, and the sum times 2^24 an integer below
// 2^36.
struct PairSums {
    double ax = 0.0, ay = 0.0;  // the terms, in 2^-30 units
    double osum = 0.0;          // the overlaps
    uint32_t worst = 0;         // the largest overlap's bits (overlaps lie in [0, 1])
    uint32_t pairs = 0;
};

// One neighbour of particle i at (dx, dy) = p_i - p_j (`other`: not i
// itself).
template <bool MOVE, bool SUMS>
__device__ __forceinline__ void stencil_visit(bool other, float dx, float dy, double &ax, double &ay,
                                              double &osum, uint32_t &worst, uint32_t &pairs) {
    float ov, F;
    if (!stencil_reach(dx, dy, other, ov, F)) return;
    worst = max(worst, __float_as_uint(ov));
    pairs += 1;
    if (SUMS) osum += (double)ov;
    if (MOVE) {
        ax += (double)rintf(dx * F);
        ay += (double)rintf(dy * F);
    }
}

// The same for a neighbour known to be within reach.
template <bool MOVE, bool SUMS>
__device__ __forceinline__ void stencil_hit(float dx, float dy, PairSums &s) {
    float sq = dx * dx;
    sq = sq + dy * dy;
    float ov, F;
    stencil_terms(sq, ov, F);
    s.worst = max(s.worst, __float_as_uint(ov));
    s.pairs += 1;
    if (SUMS) s.osum += (double)ov;
    if (MOVE) {
        s.ax += (double)rintf(dx * F);
        s.ay += (double)rintf(dy * F);
    }
}

// The 3x3 cells of a particle as the stencil kernels keep them: each row's
// first particle and length, the lengths 0 over the budget.
struct StencilRows {
    uint32_t rs[3], len[3];
    uint32_t half;  // rs[1] + half: the particle's own cell's start; kBeside: see below
};

// In StencilRows::half (at most kStencilBudget by itself): the particle lies
// beside the cell that holds it, as a loaded triple may say.  It need not be in
// the middle row then.
constexpr uint32_t kBeside = 0x8000u;
static_assert(kStencilBudget < kBeside, "half and its flag share 16 bits");

// The rows of a particle in cell k.  More than kStencilBudget particles in
// them: none, and `over` (a bound on the work of one lane).
__device__ __forceinline__ StencilRows stencil_rows_of(const FrameParams &p, const FrameBuffers &b,
                                                       uint32_t k, bool &over) {
    StencilRows r;
    const Grid g = grid_of(p, k);
    uint32_t cx, cy, own, re[3];
    cell_coords(g, k, cx, cy);
    stencil_rows(p, b, g, (int)cx, (int)cy, r.rs, re, own);
    const uint64_t total = (uint64_t)(re[0] - r.rs[0]) + (re[1] - r.rs[1]) + (re[2] - r.rs[2]);
    over = total > kStencilBudget;
#pragma unroll
    for (int t = 0; t < 3; ++t) r.len[t] = over ? 0u : re[t] - r.rs[t];
    r.half = over ? 0u : min(max(r.rs[1], own), re[1]) - r.rs[1];
    return r;
}

// A wavefront none of whose rows holds more than kShortRow particles filters
// first: four neighbours of each of the three rows at a time, their loads in
// flight together, those within reach appended to the lane's list in LDS;
// then every lane works off its list.  A loose world's lane has two or three
// neighbours a row and about half of them within reach, and the pair
// arithmetic (some 25 instructions) would otherwise run for every neighbour
// that is within reach of any of the 64 lanes, the rows one after another to
// the longest of each.  A pass over the 1M lattice is bound by these vector
// instructions: 1,065 a wavefront and 35 us with a loop per row, 690 and 21 us
// with the filter and recorded rows (the measure: 580 and 27 us, 373 and
// 14 us).  Fuller wavefronts take each row by itself: lanes of one cell then
// read the same neighbour together, and neighbours out of every lane's reach
// are skipped together: of the collapsed lattice's visits a quarter are within
// reach and 73% are within some lane's (820 us before the short rows and after;
// lists for the long ones are not tried).  kShortRow lies where the rows of a
// loose world end and those of a pile (hundreds) begin.
constexpr uint32_t kShortRow = 32;
constexpr int kHitList = 9;  // entries a lane: 18 KiB a block, 8 blocks on a CU (24 KiB, 6 blocks: 26 us)

template <bool MOVE, bool SUMS>
__device__ __forceinline__ void stencil_hits(const float2 *list, uint32_t &hits, PairSums &s) {
    for (uint32_t h = 0; __ballot(h < hits) != 0; ++h) {
        if (h < hits) {
            const float2 d = list[h * 256];
            stencil_hit<MOVE, SUMS>(d.x, d.y, s);
        }
    }
    hits = 0;
}

// The short rows of a wavefront: filter, then the list.
template <bool MOVE, bool SUMS, bool HALF>
__device__ __forceinline__ void stencil_short(const float2 *pin, uint32_t i, float xi, float yi,
                                              StencilRows r, float2 *list, PairSums &s) {
    if (HALF) {
        const uint32_t from = min(max(r.rs[1], i + 1), r.rs[1] + r.len[1]);
        r.len[1] -= from - r.rs[1];
        r.rs[1] = from;
    }
    const uint32_t longest = max(max(r.len[0], r.len[1]), r.len[2]);
    uint32_t hits = 0;
    for (uint32_t o = 0; __ballot(o < longest) != 0; o += 4) {
        // Past a row's end these are other particles, or up to three
        // entries past the last one (dmalloc's slack).
        float2 q[3][4];
#pragma unroll
        for (int t = HALF ? 1 : 0; t < 3; ++t) {
            if (o < r.len[t]) {
                const float2 *qp = pin + (r.rs[t] + o);
#pragma unroll
                for (int v = 0; v < 4; ++v) q[t][v] = qp[v];
            }
        }
#pragma unroll
        for (int t = HALF ? 1 : 0; t < 3; ++t) {
            if (__ballot(o < r.len[t]) == 0) continue;
            if (__ballot(hits > (uint32_t)kHitList - 4) != 0) stencil_hits<MOVE, SUMS>(list, hits, s);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float dx = xi - q[t][v].x, dy = yi - q[t][v].y;
                float sq = dx * dx;
                sq = sq + dy * dy;
                bool in = o + v < r.len[t];
                if (t == 1 && !HALF) in = in & (r.rs[1] + o + v != i);
                if (in & !(sq > kReachSq)) {
                    list[hits * 256] = make_float2(dx, dy);
                    ++hits;
                }
            }
        }
    }
    stencil_hits<MOVE, SUMS>(list, hits, s);
}

// Any rows, one row after another, four neighbours a step, all loaded before
// the first is used.
template <bool MOVE, bool SUMS, bool HALF>
__device__ __forceinline__ void stencil_long(const float2 *pin, uint32_t i, float xi, float yi,
                                             const uint32_t (&rs)[3], const uint32_t (&re)[3],
                                             double &ax, double &ay, double &osum, uint32_t &worst,
                                             uint32_t &pairs) {
#pragma unroll
    for (int t = HALF ? 1 : 0; t < 3; ++t) {
        uint32_t j = rs[t];
        const uint32_t e = re[t];
        for (; j + 4 <= e; j += 4) {
            // One address, four loads at constant offsets from it.
            const float2 *qp = pin + j;
            float2 q[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) q[u] = qp[u];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                stencil_visit<MOVE, SUMS>(HALF && t == 1 ? j + u > i : j + u != i, xi - q[u].x, yi - q[u].y, ax, ay,
                                          osum, worst, pairs);
        }
        for (; j < e; ++j) {
            const float2 q = pin[j];
            stencil_visit<MOVE, SUMS>(HALF && t == 1 ? j > i : j != i, xi - q.x, yi - q.y, ax, ay, osum, worst, pairs);
        }
    }
}

// Particle i at (xi, yi) against the particles of its rows: the number of
// overlapping pairs and the largest overlap, with MOVE the sum of its pair
// terms, and with SUMS the sum of the overlaps.  (A lane without a particle
// has empty rows.)  HALF: each pair once -- the later particles of its own
// cell, the cell to its right and the three cells above; every other pair of
// its 3x3 cells is one of these seen from the other particle (no particle is
// kBeside then).
template <bool MOVE, bool SUMS, bool HALF>
__device__ __forceinline__ PairSums stencil_particle(const float2 *pin, uint32_t i, float xi, float yi,
                                                     StencilRows r, float2 *list) {
    if (HALF) {
        r.len[0] = 0;
        r.rs[1] += r.half;
        r.len[1] -= r.half;
        r.half = 0;
    }
    PairSums s;
    // The short path leaves out particle i in the middle row alone;
    // stencil_long does in every row, and takes those that lie beside their
    // cell.  (Without kBeside half is at most len[1].)
    if (__ballot(max(max(r.len[0], r.len[1]), max(r.len[2], r.half)) > kShortRow) == 0) {
        stencil_short<MOVE, SUMS, HALF>(pin, i, xi, yi, r, list, s);
        return s;
    }
    double ax = 0.0, ay = 0.0, osum = 0.0;
    uint32_t worst = 0, pairs = 0;
    const uint32_t re[3] = {r.rs[0] + r.len[0], r.rs[1] + r.len[1], r.rs[2] + r.len[2]};
    stencil_long<MOVE, SUMS, HALF>(pin, i, xi, yi, r.rs, re, ax, ay, osum, worst, pairs);
    s.ax = ax;
    s.ay = ay;
    s.osum = osum;
    s.worst = worst;
    s.pairs = pairs;
    return s;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// Sum into lane 63, as wave63_max.
__device__ __forceinline__ uint32_t wave63_sum(uint32_t v) {
    v += dpp0<0x111, 0xf>(v);
    v += dpp0<0x112, 0xf>(v);
    v += dpp0<0x114, 0xf>(v);
    v += dpp0<0x118, 0xf>(v);
    v += dpp0<0x142, 0xa>(v);
    return v + dpp0<0x143, 0xc>(v);
}

// Raises word `slot` of the block's stripe to the block's largest overlap
// (its bits) -- one atomic per block that nothing waits for; with one word
// for every block they serialised, and reading it first to skip them kept
// each block resident for a memory round trip -- and, with sums, adds
// `sides` times the block's
// overlap sum (a lane's below 2^36 units of 2^-24) and pair count to its
// slot (blockIdx % kStencilSumSlots) of them.
__device__ __forceinline__ void block_report(uint32_t *words, uint32_t slot, const PairSums &s, unsigned long long *sums,
                                             unsigned long long sides) {
    __shared__ uint32_t s_max[4], s_cnt[4];
    __shared__ unsigned long long s_sum[4];
    const uint32_t wave = threadIdx.x >> 6, lane = lane_id();
    const uint32_t worst = wave63_max(s.worst);
    uint32_t cnt = 0, lo = 0, hi = 0;
    if (sums) {  // the whole grid alike
        const unsigned long long o = (unsigned long long)(s.osum * (double)kOverlapScale);
        cnt = wave63_sum(s.pairs);
        lo = wave63_sum((uint32_t)o & 0xffffffu);
        hi = wave63_sum((uint32_t)(o >> 24));
    }
    if (lane == 63) {
        s_max[wave] = worst;
        s_cnt[wave] = cnt;
        s_sum[wave] = ((unsigned long long)hi << 24) + lo;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t m = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3]));
        if (words && m) atomicMax(&words[(blockIdx.x % kWordStripes) * kWordStride + slot], m);
        const unsigned long long n = (unsigned long long)s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3];
        if (sums && n) {
            unsigned long long *to = sums + (blockIdx.x % kStencilSumSlots) * kStencilSumStride;
            atomicAdd(to, sides * (s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3]));
            atomicAdd(to + 1, sides * n);
        }
    }
}

// The particle of this lane and its rows.  The frame's first stencil kernel
// takes the particle from the lane order (StencilArgs::perm) and its cell
// from its position or from a.cell, and records both for the kernels that
// follow: a particle's 3x3 cells are the frame start's in every pass, and
// deriving the rows (a division, 21 loads and their selection) was a fifth of
// a loose pass's instructions.  Without room for the record (a.record 0) the
// first kernel leaves the cell.  A lane without a particle gets i >= p.n, or
// empty rows.
__device__ __forceinline__ StencilRows stencil_lane(const FrameParams &p, const FrameBuffers &b,
                                                    const StencilArgs &a, uint32_t &i, float2 &q) {
    StencilRows r;
#pragma unroll
    for (int t = 0; t < 3; ++t) r.rs[t] = r.len[t] = 0;
    r.half = 0;
    q = make_float2(0.0f, 0.0f);
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    i = t;
    if (t >= p.n) return r;
    if (a.rows_from == kRowsRecorded) {
        const uint4 v = a.rows[t];
        const uint2 w = a.rows2[t];
        i = w.y;
        q = a.pin[i];
        r.rs[0] = v.x;
        r.rs[1] = v.y;
        r.rs[2] = v.z;
        r.len[0] = v.w & 0xffffu;
        r.half = v.w >> 16;
        r.len[1] = w.x & 0xffffu;
        r.len[2] = w.x >> 16;
        return r;
    }
    i = a.perm ? a.perm[t] : t;
    q = a.pin[i];
    const uint32_t held = b.key[i];
    const uint32_t k = a.rows_from == kRowsOfCell ? a.cell[i] : position_key(p, particle_grid(p, b, i), q.x, q.y);
    const bool beside = k != held;
    bool over = false;
    if (k < p.ncell) r = stencil_rows_of(p, b, k, over);
    if (beside) r.half |= kBeside;
    if (beside | over) atomicOr(&a.words[kOneSidedWord], 1u);
    if (a.rows_from == kRowsOfPosition && !a.record) a.cell[i] = k;
    if (a.record) {
        a.rows[t] = make_uint4(r.rs[0], r.rs[1], r.rs[2], r.len[0] | (r.half << 16));
        a.rows2[t] = make_uint2(r.len[1] | (r.len[2] << 16), i);
    }
    return r;
}

__device__ __forceinline__ unsigned long long *stencil_sums(const StencilArgs &a) {
    return a.stat ? a.sums + (a.stat - 1) * kStencilSumSlots * kStencilSumStride : nullptr;
}

// The learned frame's fallback: whether the warm start's mean overlap
// (sums set 2) exceeds the frame start's (set 0), compared exactly as
// sum_w * n_0 > sum_0 * n_w in 128 bits.  Every block of the move computes
// it from the same words; wavefront 0 reads the 64 slots.
__device__ __forceinline__ bool warm_rejected(const StencilArgs &a) {
    __shared__ uint32_t s_rej;
    if (threadIdx.x < 64) {
        const unsigned long long *s0 = a.sums + (size_t)threadIdx.x * kStencilSumStride;
        const unsigned long long *s2 = a.sums + (size_t)(2 * kStencilSumSlots + threadIdx.x) * kStencilSumStride;
        unsigned long long v[4] = {s0[0], s0[1], s2[0], s2[1]};
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v[q] += __shfl_xor(v[q], o, 64);
        if (threadIdx.x == 0) {
            const unsigned __int128 lhs = (unsigned __int128)v[2] * v[1];
            const unsigned __int128 rhs = (unsigned __int128)v[0] * v[3];
            s_rej = lhs > rhs ? 1u : 0u;
        }
    }
    __syncthreads();
    return s_rej != 0;
}

// Whether the largest overlap recorded in word `slot` exceeds tol (overlaps
// lie in [0, 1]: the stripes' bits order as the floats).
__device__ __forceinline__ bool overlap_above(const uint32_t *words, uint32_t slot, float tol) {
    const uint32_t v = words[(lane_id() % kWordStripes) * kWordStride + slot];
    return __ballot(__uint_as_float(v) > tol) != 0;
}

// Where the positions are after passes that stop at the tolerance: pass k
// went from a.pin to a.pin_odd for even k and back for odd k, and the first
// whose start did not exceed the tolerance, if any, ended them (its output
// does not count).  The whole grid decides alike from the words.
__device__ __forceinline__ bool passes_end_odd(const StencilArgs &a) {
    static_assert(kWordStripes == 16, "four words' stripes a wavefront");
    uint32_t k = 0;
    for (bool on = true; on && k < a.select;) {
        const uint32_t v = a.words[(lane_id() & 15) * kWordStride + k + (lane_id() >> 4)];
        unsigned long long above = __ballot(__uint_as_float(v) > a.tol);
        for (int u = 0; u < 4 && on && k < a.select; ++u, above >>= 16) {
            on = (above & 0xffffull) != 0;
            k += on ? 1u : 0u;
        }
    }
    return (k & 1u) != 0;
}

// The largest overlap at positions a.pin, raised into a.words[a.in_slot]
// (non-negative floats order as their bits).  With a.pin_odd the positions
// are where the frame's a.select passes ended; with a.pout they are brought
// there.
__global__ __launch_bounds__(256, 8) void stencil_measure_kernel(FrameParams p, FrameBuffers b,
                                                              StencilArgs a) {
    __shared__ float2 s_list[kHitList * 256];
    if (a.pin_odd && passes_end_odd(a)) a.pin = a.pin_odd;
    uint32_t i;
    float2 q;
    const StencilRows r = stencil_lane(p, b, a, i, q);
    if (a.pout && a.pout != a.pin && i < p.n) a.pout[i] = q;
    const bool half = a.half && a.words[kOneSidedWord] == 0;  // the whole grid alike
    float2 *list = s_list + threadIdx.x;
    const PairSums s = half ? (a.stat ? stencil_particle<false, true, true>(a.pin, i, q.x, q.y, r, list)
                                      : stencil_particle<false, false, true>(a.pin, i, q.x, q.y, r, list))
                            : (a.stat ? stencil_particle<false, true, false>(a.pin, i, q.x, q.y, r, list)
                                      : stencil_particle<false, false, false>(a.pin, i, q.x, q.y, r, list));
    block_report(a.words, a.in_slot, s, stencil_sums(a), half ? 2ull : 1ull);
}

// The same without the measure.
__global__ __launch_bounds__(256) void stencil_end_kernel(FrameParams p, StencilArgs a) {
    if (a.pin_odd && passes_end_odd(a)) a.pin = a.pin_odd;
    if (a.pout == a.pin) return;
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < p.n) a.pout[i] = a.pin[i];
}

// One pass: a.pin -> a.pout, raising a.words[a.in_slot] to the largest
// overlap of its input.  A pass over no overlap moves nothing, so passes
// without a tolerance need no test.  With a.check the pass runs only while
// the overlap at the start of the pass before it exceeded the tolerance:
// that pass need not have run where its start did not, so the passes end at
// its start, which this one leaves alone (it would overwrite it), raising no
// overlap, so that every later pass stays away as well.  One pass too many
// costs less than a measure before each.
__global__ __launch_bounds__(256, 7) void stencil_move_kernel(FrameParams p, FrameBuffers b,
                                                           StencilArgs a) {
    __shared__ float2 s_list[kHitList * 256];
    if (a.check && !overlap_above(a.words, a.in_slot - 1, a.tol)) return;  // the whole grid
    if (a.pin_alt) {
        const bool rej = warm_rejected(a);
        if (blockIdx.x == 0 && threadIdx.x == 0) a.words[kFallbackWord] = rej ? 1u : 0u;
        if (rej) a.pin = a.pin_alt;  // a copy of the arguments: the whole grid decides alike
    }
    uint32_t i;
    float2 q;
    const StencilRows r = stencil_lane(p, b, a, i, q);
    float2 *list = s_list + threadIdx.x;
    const PairSums s = a.stat ? stencil_particle<true, true, false>(a.pin, i, q.x, q.y, r, list)
                              : stencil_particle<true, false, false>(a.pin, i, q.x, q.y, r, list);
    block_report(a.words, a.in_slot, s, stencil_sums(a), 1ull);
    if (i >= p.n) return;
    // The mean of the pair corrections (constraint averaging): a particle
    // moves at most 0.5 per pass.
    float dx = (float)s.ax * kStencilUnit;  // the integer rounded once to f32
    float dy = (float)s.ay * kStencilUnit;
    if (s.pairs > 1) {
        dx = dx / (float)s.pairs;
        dy = dy / (float)s.pairs;
    }
    a.pout[i] = make_float2(q.x + dx, q.y + dy);
}

// The frame's first stencil launch: clears the overlap words and sums, and
// sets the lane order of the separation kernels.  A pass's sums are exact
// and each lane writes its own particle, so any order gives the same result;
// this one puts the particles of each crowded cell (kCrowdMin..kCrowdMax) in
// order of x (columns of particles are the common crowd), so that the 64
// lanes of a wavefront lie close together and more of their neighbours are
// out of every lane's reach at once.
//
// One wavefront per 64 consecutive particles.  A crowded cell holds at least
// one of their starts, and the wavefront of the first of them orders it: the
// particles counted into kOrderSlices equal slices of their x range (LDS
// atomics give each its rank in its slice), the slices' starts by a
// wavefront scan, then perm over the cell's range in slice order; inside a
// slice the order is the atomics'.  Slices of 1/64 of the range are far finer
// than the 64 lanes of a wavefront need.  Every other particle keeps its
// place.  A loose 1M world takes 5 us so; clearing, listing the crowded cells
// of the whole grid and ordering them took a launch each and 15.
constexpr uint32_t kOrderSlices = 64;    // x slices of a crowded cell: one per lane
static_assert(kCrowdMin >= 64, "a crowded cell holds the start of a wavefront's particles");

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fminf(v, __shfl_xor(v, off, 64));
    return v;
}

// Positions and velocities side by side, for the features' gathers.
__global__ __launch_bounds__(256) void learn_state_kernel(const float2 *pos, const float2 *vel, float4 *state,
                                                          uint32_t n) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float2 q = pos[i], v = vel[i];
    state[i] = make_float4(q.x, q.y, v.x, v.y);
}

__global__ __launch_bounds__(256) void stencil_begin_kernel(FrameParams p, FrameBuffers b, StencilArgs a,
                                                            const float2 *pos) {
    __shared__ uint32_t slice_count[4][kOrderSlices];
    __shared__ uint32_t tag[4][kCrowdMax];  // a particle's slice << 16 | its rank in the slice
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < kWordEntries; i += gridDim.x * 256) a.words[i] = 0;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < kStencilSumSets * kStencilSumSlots; i += gridDim.x * 256) {
        a.sums[i * kStencilSumStride] = 0;
        a.sums[i * kStencilSumStride + 1] = 0;
    }
    if (!a.perm) return;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
    const uint32_t t0 = (blockIdx.x * 4 + wave) * 64, t = t0 + lane;
    if (t0 >= p.n) return;
    // The cells of this window's first particle and of the next window's: any
    // crowded cell with particles here is one of the two.
    const uint32_t k0 = b.key[t0], k1 = t0 + 64 < p.n ? b.key[t0 + 64] : kNoKey;
    uint32_t s0 = 0, e0 = 0, s1 = 0, e1 = 0;
    if (k0 < p.ncell) cell_range(p, b, k0, s0, e0);
    if (k1 < p.ncell) cell_range(p, b, k1, s1, e1);
    const uint32_t n = e0 > s0 ? e0 - s0 : 0u, n1 = e1 > s1 ? e1 - s1 : 0u;
    const bool crowd0 = n >= kCrowdMin && n <= kCrowdMax, crowd1 = n1 >= kCrowdMin && n1 <= kCrowdMax;
    const bool in0 = crowd0 && t >= s0 && t < e0, in1 = crowd1 && t >= s1 && t < e1;
    if (t < p.n && !in0 && !in1) a.perm[t] = t;
    if (!crowd0 || s0 > t0 || s0 + 64 <= t0) return;  // no crowded cell, or an earlier window's
    float lo = INFINITY, hi = -INFINITY;
    for (uint32_t r = lane; r < n; r += 64) {
        const float x = pos[s0 + r].x;
        lo = fminf(lo, x);
        hi = fmaxf(hi, x);
    }
    lo = wave_min(lo);
    hi = wave_max(hi);
    // Not finite (an infinite range): every particle in slice 0.
    const float scale = hi > lo ? (float)kOrderSlices / (hi - lo) : 0.0f;
    slice_count[wave][lane] = 0;
    wave_sync();
    for (uint32_t r = lane; r < n; r += 64) {
        // fmaxf takes 0 for a NaN; the slice is at most kOrderSlices - 1.
        const float f = fminf(fmaxf((pos[s0 + r].x - lo) * scale, 0.0f), (float)(kOrderSlices - 1));
        const uint32_t sl = (uint32_t)f;
        const uint32_t rank = atomicAdd(&slice_count[wave][sl], 1u);
        tag[wave][r] = sl << 16 | rank;
    }
    wave_sync();
    const uint32_t cnt = slice_count[wave][lane];
    wave_sync();
    slice_count[wave][lane] = wave_inclusive_sum(cnt) - cnt;
    wave_sync();
    for (uint32_t r = lane; r < n; r += 64) {
        const uint32_t g = tag[wave][r];
        const uint32_t slot = slice_count[wave][g >> 16] + (g & 0xffffu);
        if (slot < n) a.perm[s0 + slot] = s0 + r;  // always: the counts sum to n
    }
}

// ---------------------------------------------------------------------------
// Neighbour features of the learned warm start (an extension with no
// counterpart in the reference).
//
// Particle i's candidates are the other particles of the 5x5 cells around
// its cell (two cells each way, the world's own cells only), five row ranges
// of the packed layout.  It keeps the 16 nearest by (squared distance, packed
// index) -- the packed index is canonical, so the choice is unique -- and its
// feature row holds, for the r-th nearest, (x_j - x_i, y_j - y_i,
// vx_j - vx_i, vy_j - vy_i) rounded to bf16 (nearest even) at entries
// 4r..4r+3; fewer than 16 candidates leave zeros.  More than kFeatBudget
// candidates: an all-zero row (a bound on one lane's work).
//
// With a.sums it also adds the overlaps of i's pairs over the 3x3 cells
// (the pairs a separation pass visits, under the pass's budget) to the
// stencil sums, as stencil_particle does: every pair closer than 1 lies in
// the 3x3 cells, and the 3x3 ranges are tracked exactly inside the 5x5 ones.

// f32 -> bf16 bits, round to nearest even (NaN kept quiet).
__device__ __forceinline__ uint16_t bf16_bits(float f) {
    const uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

// Candidate order: key = (squared distance bits << 32) | packed index; equal
// distances are ordered by the bits of the candidates' (x, y, vx, vy) as
// unsigned integers, not by their index, so that the choice does not depend
// on the order of the particles inside a cell (two candidates equal in all
// four are interchangeable).  ~0 (no candidate) is last.
__device__ __forceinline__ bool cand_less(const float2 *pos, const float2 *vel, unsigned long long x,
                                          unsigned long long y) {
    const uint32_t hx = (uint32_t)(x >> 32), hy = (uint32_t)(y >> 32);
    if (hx != hy) return hx < hy;
    if (x == y) return false;
    const uint32_t jx = (uint32_t)x, jy = (uint32_t)y;
    const float2 px = pos[jx], py = pos[jy], vx = vel[jx], vy = vel[jy];
    const uint32_t a[4] = {__float_as_uint(px.x), __float_as_uint(px.y), __float_as_uint(vx.x),
                           __float_as_uint(vx.y)};
    const uint32_t c[4] = {__float_as_uint(py.x), __float_as_uint(py.y), __float_as_uint(vy.x),
                           __float_as_uint(vy.y)};
#pragma unroll
    for (int t = 0; t < 4; ++t)
        if (a[t] != c[t]) return a[t] < c[t];
    return false;
}

constexpr int kSortCands = 32;  // candidates ordered by the network
// A candidate's 32-bit key: its squared distance in fixed point above its
// number, for the first kKeyCands candidates.
constexpr int kNumberBits = 7;
constexpr uint32_t kKeyCands = 1u << kNumberBits;
constexpr uint32_t kDistMax = (1u << (32 - kNumberBits)) - 2;  // a key of all ones is no candidate

// Inserts candidate c into the ascending list k[0..15] (dropping the last).
// Squared distances are finite, so a real key's high word never equals the
// empty key's (0xffffffff), and cand_less reads particles only for real keys.
__device__ __forceinline__ void insert16(const float2 *pos, const float2 *vel, unsigned long long (&k)[kNbrs],
                                         unsigned long long c) {
    if (!cand_less(pos, vel, c, k[kNbrs - 1])) return;
    k[kNbrs - 1] = c;
#pragma unroll
    for (int t = kNbrs - 1; t > 0; --t) {
        const unsigned long long lo = k[t - 1], hi = k[t];
        const bool sw = cand_less(pos, vel, hi, lo);
        k[t - 1] = sw ? hi : lo;
        k[t] = sw ? lo : hi;
    }
}

// Two f32 as bf16 bits, rounded to nearest even (v_cvt_pk_bf16_f32; a NaN as
// bf16_bits keeps it).
__device__ __forceinline__ uint32_t bf16_pair(float x, float y) {
    if ((x != x) | (y != y)) return (uint32_t)bf16_bits(x) | ((uint32_t)bf16_bits(y) << 16);
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    bf16x2 v;
    v[0] = (__bf16)x;
    v[1] = (__bf16)y;
    return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ float squared_distance(float2 o, float2 q) {
    const float dx = o.x - q.x;
    const float dy = o.y - q.y;
    float sq = dx * dx;
    sq = sq + dy * dy;
    return sq;
}

// A particle's position and velocity.
__device__ __forceinline__ float4 particle_state(const FeatureArgs &a, uint32_t j) {
    if (a.state) return a.state[j];
    const float2 q = a.pos[j], v = a.vel[j];
    return make_float4(q.x, q.y, v.x, v.y);
}

// Candidate u of the list over the five rows: rows 1..4 begin at c1..c4, and
// a row's candidates lie at u + o.  (By value: a selection among array
// elements, or a closure's, became a load from scratch memory.)
__device__ __forceinline__ uint32_t candidate(uint32_t u, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t c4,
                                              uint32_t o0, uint32_t o1, uint32_t o2, uint32_t o3, uint32_t o4) {
    uint32_t o = u >= c1 ? o1 : o0;
    o = u >= c2 ? o2 : o;
    o = u >= c3 ? o3 : o;
    o = u >= c4 ? o4 : o;
    return u + o;
}

// The first kSortCands candidates are ordered in registers by Batcher's
// odd-even merge network for 32 keys, pruned to the 174 comparators that
// decide the first 17 places (select_nets.h), on 32-bit keys: the squared
// distance in 25 bits of fixed point over the largest the 5x5 cells allow,
// and the candidate's number; the next 96 are inserted into the best 17.  A
// comparator is a minimum and a maximum (on the 64-bit key of distance bits
// and packed index it was five instructions, and a wavefront inserts a few
// past the first 32 nearly always).  The order is the exact one unless two of
// the first 17 share the 25 bits: a wavefront where any lane finds that
// (hundreds do not) orders its candidates again by insertion with the exact
// comparator, as it inserts those past the first 128.
//
// 1M particles: 181 us and 4,222 vector instructions a wavefront before, now
// 118 (and 6.5 for learn_state_kernel) and 2,750.  What bounds it is the L1:
// 2,700 accesses a wavefront, most of them the 16 neighbours' gathers, one of
// 16 bytes each since positions and velocities lie side by side (two of 8
// before), and the candidates'; rows stored from each lane were 450 more.
__global__ __launch_bounds__(256, 4) void learn_features_kernel(FrameParams p, FrameBuffers b,
                                                             FeatureArgs a) {
    __shared__ union {
        uint4 rows[4][64 * 4];
        float2 list[kHitList * 256];
    } sh;
    const uint32_t lane = lane_id();
    const uint32_t lane_t = blockIdx.x * 256 + threadIdx.x;
    const bool on = lane_t < p.n;
    uint32_t i = on ? lane_t : 0u;  // a lane past the particles reads particle 0 and writes nothing
    if (on && a.perm) i = a.perm[lane_t];
    const float2 q = a.pos[i], w = a.vel[i];
    const uint32_t held = b.key[i];
    uint32_t rs[5], cum[5], m5 = 0;  // a row's first particle; candidates before its row
    StencilRows r3;
#pragma unroll
    for (int t = 0; t < 3; ++t) r3.rs[t] = r3.len[t] = 0;
    r3.half = 0;
#pragma unroll
    for (int t = 0; t < 5; ++t) rs[t] = cum[t] = 0;
    if (on) {
        const Grid g = particle_grid(p, b, i);
        uint32_t ucx, ucy;
        const uint32_t k = position_key(p, g, q.x, q.y);
        const bool cell = k != kNoKey;  // outside the grid: no candidates, a row of zeros
        cell_coords(g, cell ? k : g.base, ucx, ucy);
        const int cx = (int)ucx, cy = (int)ucy;
        const int gx = (int)g.gx, gy = (int)g.gy;
        // Per row of the 5x5 cells, its first cell and the one past its last;
        // of the 3x3 cells the same, and the own cell.  Every load is issued
        // before the first is used.
        uint32_t c[17], at[17], live[17], pre[17];
#pragma unroll
        for (int t = 0; t < 5; ++t) {
            int y = cy + t - 2;
            y = y < 0 ? 0 : y < gy ? y : gy - 1;  // a row outside the world: loaded, not used
            const uint32_t row = g.base + (uint32_t)(y * gx);
            c[2 * t] = row + (uint32_t)(cx > 1 ? cx - 2 : 0);
            c[2 * t + 1] = row + (uint32_t)(cx + 2 < gx ? cx + 3 : gx);
            if (t >= 1 && t <= 3) {
                c[8 + 2 * t] = row + (uint32_t)(cx > 0 ? cx - 1 : 0);
                c[9 + 2 * t] = row + (uint32_t)(cx + 1 < gx ? cx + 2 : gx);
            }
        }
        c[16] = k;
#pragma unroll
        for (int u = 0; u < 17; ++u) {
            const uint32_t v = c[u] < p.ncell ? c[u] : p.ncell - 1;
            live[u] = b.chunk_live[v >> kChunkShift];
            pre[u] = b.chunk_prefix[v >> kChunkShift];
            at[u] = b.idx[v + 1];  // also on large grids: FrameParams::idx_read
        }
#pragma unroll
        for (int u = 0; u < 17; ++u) {
            at[u] = offset_of(at[u], live[u], pre[u]);
            at[u] = c[u] < p.ncell && at[u] < p.n ? at[u] : p.n;
        }
        uint64_t tot5 = 0, tot3 = 0;
        uint32_t re1 = 0;
#pragma unroll
        for (int t = 0; t < 5; ++t) {
            const int y = cy + t - 2;
            const bool in = cell && y >= 0 && y < gy;  // the world's own rows only
            rs[t] = in ? at[2 * t] : 0u;
            const uint32_t re = in && at[2 * t + 1] > at[2 * t] ? at[2 * t + 1] : rs[t];
            cum[t] = (uint32_t)tot5;
            tot5 += re - rs[t];
            if (t >= 1 && t <= 3) {
                r3.rs[t - 1] = in ? at[8 + 2 * t] : 0u;
                const uint32_t e3 = in && at[9 + 2 * t] > at[8 + 2 * t] ? at[9 + 2 * t] : r3.rs[t - 1];
                r3.len[t - 1] = e3 - r3.rs[t - 1];
                tot3 += r3.len[t - 1];
                if (t == 2) re1 = e3;
            }
        }
        m5 = tot5 <= kFeatBudget ? (uint32_t)tot5 : 0u;
        const bool over = tot3 > kStencilBudget;
        r3.half = over ? 0u : min(max(r3.rs[1], at[16]), re1) - r3.rs[1];
        if (over) r3.len[0] = r3.len[1] = r3.len[2] = 0;
        const bool beside = k != held;
        if (beside) r3.half |= kBeside;
        // What the passes that follow need (stencil_lane).
        if (a.words && (beside | over)) atomicOr(&a.words[kOneSidedWord], 1u);
        if (a.rows) {
            a.rows[lane_t] = make_uint4(r3.rs[0], r3.rs[1], r3.rs[2], r3.len[0] | (r3.half << 16));
            a.rows2[lane_t] = make_uint2(r3.len[1] | (r3.len[2] << 16), i);
        } else if (a.cell) {
            a.cell[i] = k;
        }
    }
    const uint32_t c1 = cum[1], c2 = cum[2], c3 = cum[3], c4 = cum[4];
    const uint32_t o0 = rs[0], o1 = rs[1] - c1, o2 = rs[2] - c2, o3 = rs[3] - c3, o4 = rs[4] - c4;
#define WRACH_CAND(u) candidate(u, c1, c2, c3, c4, o0, o1, o2, o3, o4)
    // The 5x5 cells keep both differences below three cell sides.
    const float to_fixed = (float)(kDistMax + 2) / (18.01f * p.cs * p.cs);
    uint32_t ck[kSortCands];
#pragma unroll
    for (int u0 = 0; u0 < kSortCands; u0 += 8) {
        float sq[8];
        bool real[8];
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            const uint32_t u = (uint32_t)(u0 + v);
            uint32_t j = WRACH_CAND(u);
            j = u < m5 ? j : i;
            real[v] = j != i;
            sq[v] = squared_distance(a.pos[j], q);
        }
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            // Not finite or past the largest (no layout of the frames): the
            // largest, which two of them share.
            const uint32_t d = (uint32_t)fminf(sq[v] * to_fixed, (float)kDistMax);
            ck[u0 + v] = real[v] ? min(d, kDistMax) << kNumberBits | (uint32_t)(u0 + v) : 0xffffffffu;
        }
    }
#define WRACH_SEL_CE(x, y)                                 \
    {                                                      \
        const uint32_t lo_ = min(ck[x], ck[y]);            \
        ck[y] = max(ck[x], ck[y]);                         \
        ck[x] = lo_;                                       \
    }
    SEL_NET_32(WRACH_SEL_CE)
#undef WRACH_SEL_CE
    // Two at a time, loads together, each pushed through the best 17.
    for (uint32_t u = kSortCands; u < kKeyCands && __ballot(u < m5) != 0; u += 2) {
        uint32_t x[2];
        float sq[2];
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const uint32_t j = u + v < m5 ? WRACH_CAND(u + v) : i;
            sq[v] = squared_distance(a.pos[j], q);
            x[v] = j != i ? u + v : 0xffffffffu;
        }
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const uint32_t d = (uint32_t)fminf(sq[v] * to_fixed, (float)kDistMax);
            uint32_t c = x[v] != 0xffffffffu ? min(d, kDistMax) << kNumberBits | x[v] : 0xffffffffu;
#pragma unroll
            for (int r = 0; r <= kNbrs; ++r) {
                const uint32_t lo = min(ck[r], c);
                c = max(ck[r], c);
                ck[r] = lo;
            }
        }
    }
    bool tie = false;
#pragma unroll
    for (int r = 0; r < kNbrs; ++r) tie = tie || (ck[r + 1] != 0xffffffffu && (ck[r] ^ ck[r + 1]) < kKeyCands);
    uint32_t near[kNbrs];  // the neighbours; ~0: none
#pragma unroll
    for (int r = 0; r < kNbrs; ++r) near[r] = ck[r] != 0xffffffffu ? WRACH_CAND(ck[r] & (kKeyCands - 1)) : 0xffffffffu;
    const bool more = m5 > kKeyCands;
    if (__ballot(tie || more) != 0) {  // every lane votes
        // Lanes with a tie from their first candidate on, lanes with more
        // than kKeyCands from there on; a candidate past the 16th in fixed
        // point is past it exactly.  Two at a time, their loads in flight
        // together: one by one, positions of few bits (ties in most wavefronts:
        // 250k of 1/64 on a lattice 292 us, 229 so) and crowds (240k, 520
        // candidates each: 702 us, 544) took longer than with every candidate's
        // 64-bit key in the network (245, 562).  Four at a time spill registers
        // (158 us instead of 118 for 1M loose particles).
        const uint32_t last = ck[kNbrs - 1] >> kNumberBits;
        unsigned long long key[kNbrs];
#pragma unroll
        for (int r = 0; r < kNbrs; ++r)
            key[r] = tie || near[r] == 0xffffffffu
                         ? ~0ull
                         : ((unsigned long long)__float_as_uint(squared_distance(a.pos[near[r]], q)) << 32) | near[r];
        const uint32_t begin = tie ? 0u : kKeyCands, end = tie || more ? m5 : 0u;
        for (uint32_t u = __ballot(tie) != 0 ? 0u : kKeyCands; __ballot(u < end) != 0; u += 2) {
            uint32_t j[2];
            float sq[2];
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                j[v] = u + v >= begin && u + v < end ? WRACH_CAND(u + v) : i;
                sq[v] = squared_distance(a.pos[j[v]], q);
            }
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                if (j[v] == i) continue;
                if ((uint32_t)fminf(sq[v] * to_fixed, (float)kDistMax) > last) continue;
                insert16(a.pos, a.vel, key, ((unsigned long long)__float_as_uint(sq[v]) << 32) | j[v]);
            }
        }
#pragma unroll
        for (int r = 0; r < kNbrs; ++r)
            near[r] = (uint32_t)key[r];  // ~0 where there is none
    }
#undef WRACH_CAND
    // The rows through LDS, half a row at a time, so that a wavefront stores
    // 64 bytes of 16 rows at once (a lane's 16 bytes at a time, its stores hit
    // 64 rows each): chunk c of lane l at place c ^ (l / 2 % 4), which spreads
    // both sides over the banks.
    uint4 *out = sh.rows[threadIdx.x >> 6];
    const unsigned long long rows_on = __ballot(on);
#pragma unroll
    for (uint32_t h0 = 0; h0 < 8; h0 += 4) {
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) {
            uint32_t h[4] = {0u, 0u, 0u, 0u};
            const uint32_t n0 = near[2 * (h0 + c)], n1 = near[2 * (h0 + c) + 1];
            const float4 s0 = particle_state(a, n0 != 0xffffffffu ? n0 : i);
            const float4 s1 = particle_state(a, n1 != 0xffffffffu ? n1 : i);
            if (n0 != 0xffffffffu) {
                h[0] = bf16_pair(s0.x - q.x, s0.y - q.y);
                h[1] = bf16_pair(s0.z - w.x, s0.w - w.y);
            }
            if (n1 != 0xffffffffu) {
                h[2] = bf16_pair(s1.x - q.x, s1.y - q.y);
                h[3] = bf16_pair(s1.z - w.x, s1.w - w.y);
            }
            out[lane * 4 + (c ^ (lane >> 1 & 3))] = make_uint4(h[0], h[1], h[2], h[3]);
        }
        wave_sync();
#pragma unroll
        for (uint32_t v = 0; v < 4; ++v) {
            const uint32_t row = v * 16 + (lane >> 2), c = lane & 3;
            const uint32_t to = (uint32_t)__shfl((int)i, (int)row, 64);
            if ((rows_on >> row) & 1ull)
                reinterpret_cast<uint4 *>(a.feat + (size_t)(a.row0 + to) * kFeat)[h0 + c] =
                    out[row * 4 + (c ^ (row >> 1 & 3))];
        }
        wave_sync();
    }
    if (a.sums) {
        // The overlap sums: the 3x3 cells, as a separation pass visits them.
        __syncthreads();
        const PairSums s = stencil_particle<false, true, false>(a.pos, i, q.x, q.y, r3, sh.list + threadIdx.x);
        block_report(nullptr, 0, s, a.sums, 1ull);
    }
}

}  // namespace

// The frame launchers take optional start/stop events, which hipExtLaunchKernel
// stamps with the kernel's own start and end (wrach_step_profiled).
template <typename K>
static hipError_t launch(K kernel, uint32_t grid, uint32_t block, hipStream_t stream,
                         hipEvent_t start, hipEvent_t stop, const FrameParams &p,
                         const FrameBuffers &b) {
    if (start || stop)
        hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(block), 0, stream, start, stop, 0, p, b);
    else
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), 0, stream, p, b);
    return hipGetLastError();
}

hipError_t launch_collide(const FrameParams &p, const FrameBuffers &b, hipStream_t stream,
                          hipEvent_t start, hipEvent_t stop) {
    // One block of 4 wavefronts per 256 * kCollideWindows packed particles
    // (one block for none: the events of a profiled frame still get a kernel).
    constexpr uint32_t per_block = kCollideBlock * kCollideWindows;
    const uint32_t blocks = p.n ? (p.n + per_block - 1) / per_block : 1u;
    return launch(collide_kernel, blocks, kCollideBlock, stream, start, stop, p, b);
}

hipError_t launch_cells(const FrameParams &p, const FrameBuffers &b, hipStream_t stream,
                        hipEvent_t start, hipEvent_t stop) {
    return launch(cells_kernel, cells_blocks(b.cells_grid, p.n), kCollideBlock, stream, start, stop, p, b);
}

// Asked once per device (a frame without a context asks on every call).
uint32_t resident_blocks_cells() {
    constexpr int kDevices = 64;
    static std::atomic<uint32_t> known[kDevices];
    int dev = 0, per_cu = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (dev >= 0 && dev < kDevices)
        if (const uint32_t r = known[dev].load(std::memory_order_relaxed)) return r;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, cells_kernel, kCollideBlock, 0) != hipSuccess)
        return 0;
    const uint32_t r = (uint32_t)(per_cu > 0 ? per_cu : 1) * (uint32_t)(cus > 0 ? cus : 1);
    if (dev >= 0 && dev < kDevices) known[dev].store(r, std::memory_order_relaxed);
    return r;
}

hipError_t launch_canonical(const FrameParams &p, const FrameBuffers &b, uint32_t *idx_out, hipStream_t stream) {
    const uint32_t chunks = (p.ncell + kChunkCells - 1) / kChunkCells;
    const uint32_t blocks = (p.n + kCollideBlock - 1) / kCollideBlock;
    if (chunks + blocks == 0) return hipSuccess;
    if (relative_offsets(p.ncell)) {  // the particles' blocks read the offsets that the others would make whole
        const hipError_t e = launch_materialize(p, b, stream);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(canonical_kernel, dim3(chunks + blocks), dim3(kCollideBlock), 0, stream, p, b, idx_out);
    return hipGetLastError();
}

template <int S>
static hipError_t launch_scan_as(const FrameParams &p, const FrameBuffers &b, hipStream_t stream,
                                 hipEvent_t start, hipEvent_t stop) {
    constexpr ScanShape sh = kScanShapes[S];
    return launch(scan_kernel<sh.threads, sh.items>, b.scan_tiles, sh.threads, stream, start, stop,
                  p, b);
}

hipError_t launch_scan(const FrameParams &p, const FrameBuffers &b, hipStream_t stream,
                       hipEvent_t start, hipEvent_t stop) {
    if (relative_offsets(p.ncell)) {
        const uint32_t chunks = (p.ncell + kChunkCells - 1) / kChunkCells;
        const uint32_t per = std::min((chunks + kChipWaves - 1) / kChipWaves, kWaveChunks);
        const uint32_t cells = (chunks + 4 * per - 1) / (4 * per);
        const uint32_t tiles = (chunks + kChunkTile - 1) / kChunkTile;
        if (start || stop) {
            hipExtLaunchKernelGGL(cell_scan_kernel, dim3(cells), dim3(256), 0, stream, start, nullptr, 0, p, b, chunks,
                                  per);
            hipExtLaunchKernelGGL(chunk_scan_kernel, dim3(tiles), dim3(1024), 0, stream, nullptr, stop, 0, p, b, chunks);
        } else {
            hipLaunchKernelGGL(cell_scan_kernel, dim3(cells), dim3(256), 0, stream, p, b, chunks, per);
            hipLaunchKernelGGL(chunk_scan_kernel, dim3(tiles), dim3(1024), 0, stream, p, b, chunks);
        }
        return hipGetLastError();
    }
    static_assert(kNumScanShapes == 9, "one case per scan shape");
    switch (b.scan_shape) {
        case 8: return launch_scan_as<8>(p, b, stream, start, stop);
        case 7: return launch_scan_as<7>(p, b, stream, start, stop);
        case 6: return launch_scan_as<6>(p, b, stream, start, stop);
        case 1: return launch_scan_as<1>(p, b, stream, start, stop);
        case 2: return launch_scan_as<2>(p, b, stream, start, stop);
        case 3: return launch_scan_as<3>(p, b, stream, start, stop);
        case 4: return launch_scan_as<4>(p, b, stream, start, stop);
        case 5: return launch_scan_as<5>(p, b, stream, start, stop);
        default: return launch_scan_as<0>(p, b, stream, start, stop);
    }
}

template <int S>
static hipError_t launch_scatter_as(const FrameParams &p, const FrameBuffers &b, hipStream_t stream,
                                    hipEvent_t start, hipEvent_t stop) {
    constexpr int per = kScatterPerLane[S];
    constexpr uint32_t per_block = kScatterBlock * per;
    const uint32_t tiles = (p.n + per_block - 1) / per_block;
    const auto kernel = relative_offsets(p.ncell) ? scatter_kernel<per, true> : scatter_kernel<per, false>;
    return launch(kernel, (tiles + 7) / 8 * 8, kScatterBlock, stream, start, stop, p, b);
}

hipError_t launch_scatter(const FrameParams &p, const FrameBuffers &b, hipStream_t stream,
                          hipEvent_t start, hipEvent_t stop) {
    static_assert(kNumScatterShapes == 3, "one case per scatter shape");
    switch (b.scatter_shape) {
        case 1: return launch_scatter_as<1>(p, b, stream, start, stop);
        case 2: return launch_scatter_as<2>(p, b, stream, start, stop);
        default: return launch_scatter_as<0>(p, b, stream, start, stop);
    }
}

hipError_t launch_materialize(const FrameParams &p, const FrameBuffers &b, hipStream_t stream) {
    const uint32_t chunks = (p.ncell + kChunkCells - 1) / kChunkCells;
    if (chunks == 0) return hipSuccess;
    hipLaunchKernelGGL(materialize_kernel, dim3(chunks), dim3(256), 0, stream, p, b);
    return hipGetLastError();
}

hipError_t launch_copy32(uint32_t *dst, const uint32_t *src, size_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(copy32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, dst, src, n);
    return hipGetLastError();
}

hipError_t launch_iota(uint32_t *dst, uint32_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(iota_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, dst, n);
    return hipGetLastError();
}

hipError_t launch_keys_from_offsets(const uint32_t *idx, uint32_t ncell, uint32_t n, uint32_t *key,
                                    hipStream_t stream) {
    if (n == 0 || ncell == 0) return hipSuccess;
    hipLaunchKernelGGL(keys_from_offsets_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, idx, ncell,
                       n, key);
    return hipGetLastError();
}

hipError_t launch_noalloc_init(const FrameParams &p, const FrameBuffers &b, const uint32_t *indices,
                               hipStream_t stream) {
    const uint32_t chunks = (p.ncell + kChunkCells - 1) / kChunkCells;
    const uint32_t tiles = (p.ncell + kMinScanTile - 1) / kMinScanTile;
    if (p.ncell == 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(noalloc_init_kernel, dim3((p.ncell + 255) / 256), dim3(256), 0, stream, p, b, indices, tiles,
                       chunks);
    return hipGetLastError();
}

hipError_t launch_upload_bin(const UploadParams &u, const FrameBuffers &b, hipStream_t stream) {
    if (u.n == 0) return hipSuccess;
    hipLaunchKernelGGL(upload_bin_kernel, dim3((u.n + 255) / 256), dim3(256), 0, stream, u, b);
    return hipGetLastError();
}

hipError_t launch_outside_sum(const uint32_t *outside, uint32_t *host, hipStream_t stream) {
    hipLaunchKernelGGL(outside_sum_kernel, dim3(1), dim3(64), 0, stream, outside, host);
    return hipGetLastError();
}

hipError_t launch_store_outside_count(const UploadParams &u, uint32_t *counts, hipStream_t stream) {
    if (u.n == 0) return hipSuccess;
    hipLaunchKernelGGL(store_outside_count_kernel, dim3((u.n + 255) / 256), dim3(256), 0, stream, u,
                       counts);
    return hipGetLastError();
}

hipError_t launch_store_outside(const UploadParams &u, float2 *dpos, float2 *dvel, uint32_t base,
                                const uint32_t *offsets, hipStream_t stream) {
    if (u.n == 0) return hipSuccess;
    hipLaunchKernelGGL(store_outside_kernel, dim3((u.n + 255) / 256), dim3(256), 0, stream, u, dpos,
                       dvel, base, offsets);
    return hipGetLastError();
}

hipError_t launch_upload_scatter(const UploadParams &u, const FrameBuffers &b, hipStream_t stream) {
    const uint32_t blocks = u.n ? (u.n + 255) / 256 : 1;  // block 0 advances the epoch
    hipLaunchKernelGGL(upload_scatter_kernel, dim3(blocks), dim3(256), 0, stream, u, b);
    return hipGetLastError();
}

hipError_t launch_stencil_measure(const FrameParams &p, const FrameBuffers &b, const StencilArgs &a,
                                  hipStream_t stream) {
    if (p.n == 0) return hipSuccess;
    hipLaunchKernelGGL(stencil_measure_kernel, dim3((p.n + 255) / 256), dim3(256), 0, stream, p, b, a);
    return hipGetLastError();
}

hipError_t launch_stencil_end(const FrameParams &p, const StencilArgs &a, hipStream_t stream) {
    if (p.n == 0 || (!a.pin_odd && a.pin == a.pout)) return hipSuccess;
    hipLaunchKernelGGL(stencil_end_kernel, dim3((p.n + 255) / 256), dim3(256), 0, stream, p, a);
    return hipGetLastError();
}

hipError_t launch_stencil_move(const FrameParams &p, const FrameBuffers &b, const StencilArgs &a,
                               hipStream_t stream) {
    if (p.n == 0) return hipSuccess;
    hipLaunchKernelGGL(stencil_move_kernel, dim3((p.n + 255) / 256), dim3(256), 0, stream, p, b, a);
    return hipGetLastError();
}

hipError_t launch_learn_features(const FrameParams &p, const FrameBuffers &b, const FeatureArgs &a,
                                 hipStream_t stream) {
    if (p.n == 0) return hipSuccess;
    if (a.state) {
        hipLaunchKernelGGL(learn_state_kernel, dim3((p.n + 255) / 256), dim3(256), 0, stream, a.pos, a.vel, a.state,
                           p.n);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(learn_features_kernel, dim3((p.n + 255) / 256), dim3(256), 0, stream, p, b, a);
    return hipGetLastError();
}

hipError_t launch_stencil_begin(const FrameParams &p, const FrameBuffers &b, const StencilArgs &a,
                                const float2 *pos, hipStream_t stream) {
    const uint32_t blocks = p.n ? (p.n + 255) / 256 : 1u;
    hipLaunchKernelGGL(stencil_begin_kernel, dim3(blocks), dim3(256), 0, stream, p, b, a, pos);
    return hipGetLastError();
}

hipError_t launch_check_pair_arithmetic(unsigned long long *out, hipStream_t stream) {
    hipLaunchKernelGGL(check_pair_arithmetic_kernel, dim3(4096), dim3(256), 0, stream, out);
    return hipGetLastError();
}

}  // namespace wrach
