// resident.h -- Jacobi iterations of a cell grid in one launch whose blocks
// stay resident (the Darcy pressure solve and the Navier-Stokes epsilon).
//
// What bounds a sweep launched by itself is the launch: on 48 x 48 x 96 cells
// the arithmetic and the traffic of one sweep take about 1 us, the dependent
// launch 5.5 us (Darcy) and 6.8 us (Navier-Stokes); here an iteration takes
// 2.3 us, and 1.6 us on 15 x 15 x 44 cells (4.4 to 5.5 us launched), of which
// the trip of the halo values through memory is about 1.3 us.  The grid is divided
// into at most one tile per compute unit; a tile's iterate lies in LDS and
// registers, the constants of its cells in registers, for all iterations of
// the launch.  Per iteration a block posts the values of its tile's outer
// cells in its outbox and reads its halo from its neighbours' outboxes.
//
// There is no grid barrier.  An outbox word carries half of an FP64 value and
// the iteration's tag in one 64-bit relaxed agent-scope atomic, so a reader
// polls the data itself: one trip through memory per iteration, no fence, no
// cache write-back.  Two generations suffice: a tile writes iteration
// it + 2 only after it has read its neighbours' it + 1, which they write only
// after they have read its it.
//
// Convergence: every tenth iteration each block posts its largest residual;
// one wave per block, which owns no cells, gathers all blocks' posts three
// iterations later, so the gather overlaps the iterations, and every block
// reaches the same verdict from the same words.  A converged solve takes the
// values kept at the tested iteration; the up to three iterations past it are
// dropped.
//
// Every wait is bounded (`spin` polls).  A wait that runs out marks the solve
// state RES_ABORT, every block then leaves, and the host repeats the solve
// with one launch per sweep.  Blocks of one launch need to be resident
// together: the grid is at most one block per compute unit, and
// resident_begin() and resident_end() let the resident launches of a device
// follow each other.  The grid barriers of the list rebuild (k_rebuild,
// k_rebuild_lists, k_rebuild_multi) need the same of their blocks, and a compute
// unit that holds a block of 1024 threads at 104 registers has room for one
// block of theirs: partly placed, the two kinds could keep each other's rest
// out until a bound runs out.  So both are never in flight together: a call
// that may enqueue rebuilds holds a BarrierUse, whose stream waits for the last
// resident launch, and while one is held elsewhere a solve takes one launch
// per sweep.  Another process on the card is not seen: there the bound ends
// the wait.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "multi.h"

#define RES_ABORT 3u          // solve state: a wait ran out, nothing of the launch is valid
#define RES_SPIN (1u << 20)   // default bound of a wait in polls (about 1 s)
#define RES_CELL_THREADS 960  // threads owning cells: a block's 1024 less the gathering wave
#define RES_CHECK 10u         // iterations between residual tests
#define RES_CHUNK 20000u      // iterations of a launch at most: some 30 ms
#define RES_LAG 3u            // iterations between a test and its verdict
// The wait before a wave reads its halo, in units of 4 cycles: longer by
// RES_MORE after an iteration in which a value came late, else shorter by
// RES_LESS, so that about one iteration in five reads twice.  On 48 x 48 x 96
// cells the reads of 256 blocks that poll without a wait slow the posts down:
// 3.9 us per iteration, 2.3 with the wait.  A ratio of 8 gains another 2%; at
// 16 the waits of neighbouring blocks drive each other up (4 us).
#define RES_MORE 8u
#define RES_LESS 2u
#define RES_WAIT_MAX 512u

struct ResidentArgs {
    int n[3];   // interior cells per axis
    int T[3];   // tiles per axis
    int wrap;   // bit k: axis k is periodic
    uint32_t it0, it1;  // iterations [it0, it1)
    uint32_t tag0;      // tag of iteration it0
    uint32_t box;       // outbox words per generation and half: the largest shell
    uint32_t spin;
    unsigned long long *mail;   // [tile][2 generations][box][2 halves]
    unsigned long long *slots;  // [2 generations][tiles][2 halves]
};

// Host side (resident.hip): the division of a grid into tiles, the outboxes.
struct Resident {
    int T[3] = {0, 0, 0};
    int wrap = 0;
    uint32_t tiles = 0, threads = 0, per_thread = 0, lds = 0, box = 0;
    size_t words = 0;                     // outbox and slot words
    unsigned long long *words_d = nullptr;
    uint32_t tag = 1;                     // next unused tag
    bool usable = false;                  // false: one launch per sweep
    bool planned = false;
    uint32_t rest = 0;                    // solves left to launches per sweep after a wait ran out
    uint32_t pause = 0;                   // their number after the last such wait
    uint64_t solves = 0;                  // solves whose result came from resident launches
    uint64_t repeated = 0;                // solves in which a wait ran out
    uint64_t yielded = 0;                 // solves left to launches per sweep by a BarrierUse
};
// The bound of the waits of the launches that begin at iteration `from` or
// later, in polls (0: RES_SPIN, as for the others).
struct ResidentWait {
    uint32_t polls = 0, from = 0;
};
// Chooses the tiles of an nx x ny x nz grid on this device; usable stays false
// where the grid does not fit (see resident.hip).
void resident_plan(Resident &r, int device, int nx, int ny, int nz, int wrap);
void resident_free(Resident &r);
// The next solve is to run in resident launches.
bool resident_ready(Resident &r);
// A wait ran out: the next 16 solves, and twice as many after each further such
// wait, are left to launches per sweep (what kept a block out, another process
// on the card for instance, may have gone by then, and a wait costs a second).
void resident_gave_up(Resident &r);
// The arguments of one launch over iterations [it0, it1); false if the outboxes
// could not be made.
bool resident_args(Resident &r, hipStream_t s, int nx, int ny, int nz, uint32_t it0, uint32_t it1,
                   const ResidentWait &wait, ResidentArgs &out);
// Resident launches of one device wait for each other: call before and after
// the launch.  False, and then no launch: a BarrierUse of the device is held,
// beside `held` that the caller itself holds for stream s.
bool resident_begin(int device, hipStream_t s, uint32_t held);
void resident_end(int device, hipStream_t s);

// Held while stream s of a device may run grid barriers.
class BarrierUse {
public:
    BarrierUse() = default;
    BarrierUse(const BarrierUse &) = delete;
    BarrierUse &operator=(const BarrierUse &) = delete;
    ~BarrierUse() { close(); }
    void open(int device, hipStream_t s);
    void close();  // waits for the stream first

private:
    int device_ = -1;
    hipStream_t stream_ = nullptr;
};

#if defined(__HIPCC__)

__device__ __forceinline__ void res_barrier()
{
    // only LDS is shared across the barrier: global stores stay in flight
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Both halves go out in one 16-byte agent-scope store (two 8-byte stores 16
// bytes apart per lane took 20% longer per iteration on 48 x 48 x 96 cells).
typedef uint32_t res_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void res_post(unsigned long long *w, uint32_t tag, double v)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const res_u32x4 q = {(uint32_t)b, tag, (uint32_t)(b >> 32), tag};
    // the no-ops: a store reads its data registers within two cycles of issue
    asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" : : "v"(w), "v"(q) : "memory");
}

// Waits for the value tagged `tag`; false once the bound is reached or another
// block gave up (state holds RES_ABORT).  Both halves come in one 16-byte
// agent-scope load: each half carries the tag, so it does not matter whether
// the halves are read at one moment.
template <typename S>
__device__ __forceinline__ bool res_wait(const unsigned long long *w, uint32_t tag, uint32_t spin,
                                         const S *state, unsigned long long &bits, uint32_t &k)
{
    for (k = 0;; ++k) {
        res_u32x4 q;
        asm volatile("global_load_dwordx4 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)"
                     : "=&v"(q)
                     : "v"(w)
                     : "memory");
        if (q.y == tag && q.w == tag) {
            bits = (unsigned long long)q.x | ((unsigned long long)q.z << 32);
            return true;
        }
        if (k >= spin) return false;
        if ((k & 63u) == 63u &&
            __hip_atomic_load(state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (S)RES_ABORT)
            return false;
    }
}

// The cells of a tile are numbered shell first: the two z faces, the y faces
// between them, the x faces between those, then the inside, so that the
// posted cells belong to the first waves and a tile's outbox is written as
// one run.  A tile with an axis of up to two cells is all shell.
__host__ __device__ inline int res_shell(const int e[3])
{
    if (e[0] <= 2 || e[1] <= 2 || e[2] <= 2) return e[0] * e[1] * e[2];
    return e[0] * e[1] * e[2] - (e[0] - 2) * (e[1] - 2) * (e[2] - 2);
}

__device__ __forceinline__ void res_cell(const int e[3], int i, int &x, int &y, int &z)
{
    if (e[0] <= 2 || e[1] <= 2 || e[2] <= 2) {
        x = i % e[0], y = (i / e[0]) % e[1], z = i / (e[0] * e[1]);
        return;
    }
    const int fz = e[0] * e[1], fy = e[0] * (e[2] - 2), fx = (e[1] - 2) * (e[2] - 2);
    if (i < 2 * fz) {
        z = i < fz ? 0 : e[2] - 1;
        if (i >= fz) i -= fz;
        x = i % e[0], y = i / e[0];
        return;
    }
    i -= 2 * fz;
    if (i < 2 * fy) {
        y = i < fy ? 0 : e[1] - 1;
        if (i >= fy) i -= fy;
        x = i % e[0], z = 1 + i / e[0];
        return;
    }
    i -= 2 * fy;
    if (i < 2 * fx) {
        x = i < fx ? 0 : e[0] - 1;
        if (i >= fx) i -= fx;
        y = 1 + i % (e[1] - 2), z = 1 + i / (e[1] - 2);
        return;
    }
    i -= 2 * fx;
    x = 1 + i % (e[0] - 2);
    y = 1 + (i / (e[0] - 2)) % (e[1] - 2);
    z = 1 + i / ((e[0] - 2) * (e[1] - 2));
}

// the number of shell cell (x, y, z), the inverse of res_cell
__device__ __forceinline__ int res_shell_index(const int e[3], int x, int y, int z)
{
    if (e[0] <= 2 || e[1] <= 2 || e[2] <= 2) return x + e[0] * (y + e[1] * z);
    const int fz = e[0] * e[1], fy = e[0] * (e[2] - 2), fx = (e[1] - 2) * (e[2] - 2);
    if (z == 0 || z == e[2] - 1) return (z == 0 ? 0 : fz) + x + e[0] * y;
    if (y == 0 || y == e[1] - 1) return 2 * fz + (y == 0 ? 0 : fy) + x + e[0] * (z - 1);
    return 2 * fz + 2 * fy + (x == 0 ? 0 : fx) + (y - 1) + (e[1] - 2) * (z - 1);
}

// n / d for a fixed divisor, correctly rounded: with rh = 1 / d rounded and rl
// the rest of 1 / d, q = n rh + n rl is within one unit in the last place of
// n / d, and one correction by its exact remainder then rounds correctly
// (Markstein's theorem).  Four operations in place of the general division's
// eleven.  It holds while nothing over- or underflows: a value past 1e300
// comes out not finite, and the caller then divides.
struct FixedDiv {
    double d, rh, rl;
};
inline FixedDiv fixed_div(double d)
{
    FixedDiv f;
    f.d = d;
    f.rh = 1.0 / d;
    f.rl = __builtin_fma(-d, f.rh, 1.0) / d;
    return f;
}
template <bool FIXED>
__device__ __forceinline__ double div_by(double n, const FixedDiv &f)
{
    if (!FIXED) return n / f.d;
    const double q = __builtin_fma(n, f.rh, n * f.rl);
    return __builtin_fma(__builtin_fma(-f.d, q, n), f.rh, q);
}

// Op: the equations of one cell.
//   typedef State;                    type of the solve-state word
//   State *state() const;             0 running, else the solve has ended
//   double in(x, y, z) const;         the iterate at it0
//   struct Cell; void load(Cell &, x, y, z) const;
//   double step(Cell &, p, xn, xp, yn, yp, zn, zp, check, bits) const;
//                                     next value; bits: |residual| pattern
//   unsigned verdict(bits, it) const; 0 go on, 1 converged, 2 NaN
//   void record(bits, it, verdict) const;  one thread of the launch
//   void finish(x, y, z, value, previous) const;
template <class Op, int CPT>
__global__ void __launch_bounds__(1024) k_resident_jacobi(ResidentArgs r, Op op)
{
    extern __shared__ double res_lds[];
    __shared__ unsigned long long s_part[16];
    __shared__ unsigned s_ctl[3];  // by iteration parity, and after the last: 0, 1, 2 or RES_ABORT
    const uint32_t tid = threadIdx.x, nth = blockDim.x - 64u;  // the last wave owns no cells
    const bool aux = tid >= nth;
    // the solve ended in an earlier launch (a verdict of this launch needs
    // every block's post, so no block can read one here)
    if (tid == 0) s_ctl[0] = *(volatile typename Op::State *)op.state() != 0 ? 1u : 0u;
    res_barrier();
    if (*(volatile unsigned *)&s_ctl[0]) return;
    const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
    int t[3], x0[3], e[3];
    t[0] = (int)(tile % (uint32_t)r.T[0]);
    t[1] = (int)((tile / (uint32_t)r.T[0]) % (uint32_t)r.T[1]);
    t[2] = (int)(tile / (uint32_t)(r.T[0] * r.T[1]));
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        x0[a] = t[a] * r.n[a] / r.T[a];
        e[a] = (t[a] + 1) * r.n[a] / r.T[a] - x0[a];
    }
    const int cells = e[0] * e[1] * e[2], shell = res_shell(e);
    const int sy = e[0] + 2, sz = sy * (e[1] + 2), vol = sz * (e[2] + 2);
    if (tid == 0) s_ctl[1] = s_ctl[2] = 0u;

    typename Op::Cell cell[CPT];
    double v[CPT], prev[CPT], snap[CPT];
    int li[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        const int i = (int)tid + k * (int)nth;
        li[k] = -1;
        v[k] = prev[k] = snap[k] = 0.0;
        if (aux || i >= cells) continue;
        int x, y, z;
        res_cell(e, i, x, y, z);
        li[k] = (x + 1) + sy * (y + 1) + sz * (z + 1);
        v[k] = op.in(x0[0] + x, x0[1] + y, x0[2] + z);
        op.load(cell[k], x0[0] + x, x0[1] + y, x0[2] + z);
        res_lds[(r.it0 & 1u) * vol + li[k]] = v[k];
    }
    // the halo values this thread reads: LDS index and word of the owner's outbox
    int hl[CPT], hw[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        int h = (int)tid + k * (int)nth;
        hl[k] = hw[k] = -1;
        if (aux) h = 1 << 30;
#pragma unroll
        for (int d = 0; d < 6; ++d) {  // -x, +x, -y, +y, -z, +z
            constexpr int B[3] = {1, 0, 0}, C[3] = {2, 2, 1};
            const int a = d >> 1, b = B[a], c = C[a];
            int q = t[a] + ((d & 1) ? 1 : -1);
            const bool edge = q < 0 || q >= r.T[a];
            if (edge) q = q < 0 ? r.T[a] - 1 : 0;
            const int face = edge && !((r.wrap >> a) & 1) ? 0 : e[b] * e[c];  // 0: a boundary of the grid
            if (h >= 0 && h < face) {
                int at[3], own[3], o[3], en[3], tn[3];
                at[b] = own[b] = h % e[b];
                at[c] = own[c] = h / e[b];
                at[a] = (d & 1) ? e[a] : -1;
                o[b] = x0[b], o[c] = x0[c], o[a] = q * r.n[a] / r.T[a];
                en[b] = e[b], en[c] = e[c], en[a] = (q + 1) * r.n[a] / r.T[a] - o[a];
                tn[b] = t[b], tn[c] = t[c], tn[a] = q;
                own[a] = (d & 1) ? 0 : en[a] - 1;
                hl[k] = (at[0] + 1) + sy * (at[1] + 1) + sz * (at[2] + 1);
                hw[k] = (tn[0] + r.T[0] * (tn[1] + r.T[1] * tn[2])) * 4 * (int)r.box +
                        2 * res_shell_index(en, own[0], own[1], own[2]);
                res_lds[(r.it0 & 1u) * vol + hl[k]] = op.in(o[0] + own[0], o[1] + own[1], o[2] + own[2]);
            }
            h -= face;
        }
    }
    res_barrier();

    unsigned long long *outbox = r.mail + (size_t)tile * 4u * r.box;
    const bool shell_wave = !aux && (int)(tid & ~63u) < shell;
    const uint32_t nblk = gridDim.x;
    uint32_t chk = 0u;      // the tested iteration whose verdict is open
    bool open = false;
    unsigned ended = 0u;
    uint32_t wait = 0u;     // before the halo is read, units of 4 cycles
    // the gathering wave: every block's largest residual of iteration chk
    auto gather = [&](unsigned *ctl) {
        const uint32_t tag = r.tag0 + (chk - r.it0);
        const unsigned long long *w = r.slots + (size_t)((chk / RES_CHECK) & 1u) * 2u * nblk;
        unsigned long long m = 0ull;
        bool ok = true;
        for (uint32_t b = tid - nth; b < nblk && ok; b += 64u) {
            unsigned long long q = 0ull;
            uint32_t reads;
            ok = res_wait(w + 2u * b, tag, r.spin, op.state(), q, reads);
            m = q > m ? q : m;
        }
        ok = __all(ok);
        for (int o = 32; o > 0; o >>= 1) {
            const unsigned long long q = __shfl_xor(m, o, 64);
            m = q > m ? q : m;
        }
        if (tid == nth) {
            if (!ok) {
                *ctl = RES_ABORT;
                atomicMax(op.state(), (typename Op::State)RES_ABORT);
            } else {
                const unsigned c = op.verdict(m, chk);
                if (tile == 0) op.record(m, chk, c);
                if (c) *ctl = c;
            }
        }
    };
    for (uint32_t it = r.it0; it < r.it1; ++it) {
        const double *cur = res_lds + (it & 1u) * vol;
        double *nxt = res_lds + ((it + 1u) & 1u) * vol;
        const uint32_t tag = r.tag0 + (it - r.it0);
        const bool check = it % RES_CHECK == 0u;
        const int gen = (int)((it & 1u) * 2u * r.box);
        if (!aux) {
            bool late = false;
            // the waves whose cells the neighbours wait for go first
            if (shell_wave) __builtin_amdgcn_s_setprio(3);
            unsigned long long bits = 0ull;
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                if (li[k] < 0) continue;
                const int l = li[k];
                unsigned long long q = 0ull;
                prev[k] = v[k];
                v[k] = op.step(cell[k], v[k], cur[l - 1], cur[l + 1], cur[l - sy], cur[l + sy], cur[l - sz],
                               cur[l + sz], check, q);
                nxt[l] = v[k];
                if ((int)tid + k * (int)nth < shell) res_post(outbox + gen + 2u * (tid + k * nth), tag, v[k]);
                if (check) {
                    snap[k] = v[k];
                    bits = q > bits ? q : bits;
                }
            }
            if (shell_wave) __builtin_amdgcn_s_setprio(0);
            // first read when the neighbours' values are due: reading earlier
            // only loads the fabric the values travel on
            for (uint32_t q = 0; q < wait / 16u; ++q) __builtin_amdgcn_s_sleep(1);
            if (check) {
                for (int o = 32; o > 0; o >>= 1) {
                    const unsigned long long q = __shfl_xor(bits, o, 64);
                    bits = q > bits ? q : bits;
                }
                if ((tid & 63u) == 0u) s_part[tid >> 6] = bits;
            }
#pragma unroll
            for (int k = 0; k < CPT; ++k) {
                if (hl[k] < 0) continue;
                unsigned long long q = 0ull;
                uint32_t reads = 0u;
                if (res_wait(r.mail + hw[k] + gen, tag, r.spin, op.state(), q, reads)) {
                    if (k == 0) late = reads > 0u;
                    nxt[hl[k]] = __longlong_as_double((long long)q);
                } else {
                    s_ctl[it & 1u] = RES_ABORT;
                    atomicMax(op.state(), (typename Op::State)RES_ABORT);
                }
            }
            wait = __any(late) ? wait + RES_MORE : wait > RES_LESS ? wait - RES_LESS : 0u;
            if (wait > RES_WAIT_MAX) wait = RES_WAIT_MAX;
        } else if (open && it == chk + RES_LAG) {
            gather(&s_ctl[it & 1u]);
        }
        res_barrier();
        // a word of s_ctl that is not 0 ends every thread here, so it never
        // needs clearing; the next iteration writes the other word
        ended = *(volatile unsigned *)&s_ctl[it & 1u];
        if (ended) break;
        if (open && it == chk + RES_LAG) open = false;
        if (check) {
            if (aux) {
                unsigned long long m = 0ull;
                for (uint32_t w = 0; w < nth / 64u; ++w) m = s_part[w] > m ? s_part[w] : m;
                if (tid == nth)
                    res_post(r.slots + ((size_t)((it / RES_CHECK) & 1u) * nblk + tile) * 2u, tag,
                             __longlong_as_double((long long)m));
            }
            chk = it;
            open = true;
        }
    }
    if (!ended && open) {
        if (aux) gather(&s_ctl[2]);
        res_barrier();
        ended = *(volatile unsigned *)&s_ctl[2];
    }
    if (ended == RES_ABORT || aux) return;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        if (li[k] < 0) continue;
        int x, y, z;
        res_cell(e, (int)tid + k * (int)nth, x, y, z);
        op.finish(x0[0] + x, x0[1] + y, x0[2] + z, ended ? snap[k] : v[k], prev[k]);
    }
}

// false: not now (resident_begin)
template <class Op>
bool resident_launch(const Resident &r, int device, hipStream_t s, const ResidentArgs &a, const Op &op,
                     uint32_t held = 0u)
{
    if (!resident_begin(device, s, held)) return false;
    if (r.per_thread == 1)
        hipLaunchKernelGGL((k_resident_jacobi<Op, 1>), dim3(r.tiles), dim3(r.threads), r.lds, s, a, op);
    else
        hipLaunchKernelGGL((k_resident_jacobi<Op, 2>), dim3(r.tiles), dim3(r.threads), r.lds, s, a, op);
    resident_end(device, s);
    return true;
}

#endif
