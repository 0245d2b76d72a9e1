// resident2d.hip -- the 2D time loop with the wavefield held on the chip.
//
// The step kernels of cda2d.hip move every field through memory once per time
// step and are bound by that traffic (25.5 us per forward and 39.5 us per
// adjoint step of 16 shots of 1041 x 341 nodes, FP32, order 8) or, where the
// fields are small, by the launch of every step (6.4 us for 77 x 67 nodes).
// Shots are independent and a shot's fields are small, so here a launch keeps
// them in registers and LDS for hundreds of steps: only the forward history
// (dWaveOp, written or read once per step), the receivers' nodes and the rows
// at strip borders move.  Now 17.3 and 19.8 us for the 16 shots, 3.0 us for
// the small one.  With few strips the exchange of border rows bounds a step;
// with many the waves of the PML rows, by their vector instructions (all SIMDs
// together issue them in 57 % of the cycles) and their waits (56 % of a wave's
// cycles; the LDS is busy in 18 %, bank conflicts 5 %).
//
// Split: a shot is cut along x into strips of whole rows, one 512-thread
// workgroup per strip, one workgroup per CU.  u of the strip (and Phi where
// it can be nonzero) sits in LDS, padded by `order/2` rows above and below
// and by whole 16-byte cells left and right, so stencils need no bounds
// checks.  A thread owns one 16-byte cell column (4 FP32 or 2 FP64 nodes
// along z) over up to kPlainRows rows (kFullRows where the PML update is
// needed) and keeps du, C^2 and, backward, the imaging sums and the next
// step's history values in registers.  Waves are of one kind: plain nodes or
// PML nodes.  A step is a march of every thread along x through its rows with
// a register window, reading the z neighbour cells from LDS; u_{k+1} goes to
// the other of two LDS copies of the strip, so a step has one barrier.
//
// Rows at a strip's border go to the neighbouring strip through device
// memory, in jobs of 64 columns: the writer stores them past its caches
// (agent-coherent stores), waits for them, and stores the step's tag next to
// them; the reader polls the tag and loads the cells past its caches.
// There is no barrier across the grid (2.3-20 us per step); an exchange takes
// about 2 us, most of it under the march of the inner rows.  Two buffers
// alternate: a strip writes step k + 2 only after it has read step k + 1,
// which its neighbour publishes after reading step k.  The exchange, the
// receivers and the sources belong to waves that compute nothing: memory
// operations return in order, so a wave that polls would wait for its own
// history loads and stores as well.  They fill the border rows in LDS and
// count them there; the marches end at the borders and look at the counts
// only there.  A memory operation of this kind takes a CU about 60 cycles
// whatever its width, hence whole cells: 64-bit words with a tag in each
// need no second round trip but four times the operations, and took 3.5 us
// instead of 2.4 for 341 FP32 nodes of order 8.
//
// All strips of a launch must run at the same time (a cooperative launch of
// at most one workgroup per CU).  Every poll is bounded.  One that reaches the
// bound ends its strip, whose neighbours' polls then expire in turn, and sets
// `err` and `stop`; strips of other shots run on.  Launches that find `stop`
// set take no step.  The stopped strips leave NaN in the state, and
// resident_seal, queued behind the runs, turns the traces and the image of the
// whole batch into NaN.
//
// The arithmetic is that of cda2d.hip's batch steps, operation by operation,
// so results equal the step loop's bit for bit.
#include "common.h"

#include <algorithm>
#include <vector>

#pragma clang fp contract(off)

namespace pa {

constexpr int kResThreads = 512;
// rows of a thread's cell column: registers for du, C^2, the imaging sums and
// the prefetched history (16 B per row each) plus the march's window fill the
// 256 VGPRs that two waves per SIMD leave.  PML rows: with 7 the FP32 adjoint
// spilled 18 registers, 23.7 us a step of 16 shots of 1041 x 341 nodes of
// order 8; with 6 (2 spilled) 20.3, with 5 (none) 20.3 and the forward with
// its store 18.7 instead of 19.4.
constexpr int kPlainRows = 9;
constexpr int kFullRows = 5;
constexpr int kStripInts = 32;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct CellOf { static constexpr int V = 16 / (int)sizeof(T); };

// one 16-byte cell: V nodes along z
template <typename T>
struct alignas(16) Cell {
    T v[CellOf<T>::V];
};

template <typename T>
struct ResParams {
    AxisCoef<T> cx, cz;
    TimeCoef<T> tc;
    const int *strips;    // kStripInts per strip
    const int4 *items;    // per kind of strip and thread {row base, flags, own rows | first row << 16 | late << 24, column | thread it repeats << 16}
    const int2 *finfo;    // per strip with sources and thread {first source cell, rows with sources}
    const int *inj_lds;   // per source node: element offset in the source cells
    const int *rec_lds;   // per receiver node: byte offset in LDS
    const T *pre;         // source values, slot-major
    T *recbuf;            // receiver node values, slot-major
    char *xchg;
    long long xstride;    // bytes per strip
    int xcells;           // cells of one border and time level
    int *err;             // host word and, for the launches behind this one, device word of an expired wait
    int *stop;
    unsigned epoch;
    int strip0, slot_begin, n_steps, direction, seg_base;
    int n_inj, n_rec, adjoint_tables, record, window, spin;
};

// item flags: march towards -x; the border rows it needs from its first or
// only from its last rows on; kind in bits 3-4: 0 idle, 1 plain, 2 full, 3 exchange
enum { I_REV = 1, I_BEGIN_TOP = 2, I_BEGIN_BOT = 4, I_KIND = 8, I_END_TOP = 32, I_END_BOT = 64 };
enum { S_XTYPE = 1, S_PXTOP = 2, S_PXBOT = 4 };

// an LDS word another wave writes: an atomic load, which stays one LDS access
// (a volatile one goes through the flat path)
__device__ __forceinline__ int lds_word(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <typename T> __device__ __forceinline__ Cell<T> lds_cell(const char *smem, int off)
{
    return __builtin_bit_cast(Cell<T>, *reinterpret_cast<const u32x4 *>(smem + off));
}
template <typename T> __device__ __forceinline__ void lds_put(char *smem, int off, const Cell<T> &c)
{
    *reinterpret_cast<u32x4 *>(smem + off) = __builtin_bit_cast(u32x4, c);
}
template <typename T, bool NT = false> __device__ __forceinline__ Cell<T> cell_ld(Rsrc r, int off)
{
    return __builtin_bit_cast(Cell<T>, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, NT ? 2 : 0));
}
template <typename T, bool NT = false> __device__ __forceinline__ void cell_st(Rsrc r, int off, const Cell<T> &c)
{
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, c), r, off, 0, NT ? 2 : 0);
}

// what a thread needs besides its register arrays
template <typename T, int R>
struct ResCtx {
    static constexpr int V = CellOf<T>::V;
    static constexpr int HC = (R + V - 1) / V;  // halo cells on each side of a row
    char *smem;
    int *bad;
    int ub, ustep;        // LDS byte offset of row j = 0's cell, bytes per row of the march
    int pxb, pxstep, pzb, pzstep;
    int uw, pxw2, pzw2;   // from the copy a step reads to the one it writes
    int gb, gstep;        // byte offset in a field of the shot of row j = 0, bytes per row
    int own, first;       // rows this thread owns (bit per j), first row of the wave
    bool late;            // the wave's first row is not this thread's
    int drop;             // LDS byte offset of a cell nobody reads
    int rbase, dir, nr, col;
    int flags;            // item flags
    int lwb, pxw;         // bytes per LDS row of u and Phix
    int fany;             // rows where any lane of the wave has a source
    int flag;             // LDS byte offset of the border rows' counts
    int want_top, want_bot;  // their values once this step's rows are there
};

// Row addresses and masks are invariant over the time loop: hoisted out of it
// they would take more registers than the fields.  Values passed through here
// are recomputed from where they are used.
__device__ __forceinline__ void vfresh(int &x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void vfresh(float &x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void vfresh(double &x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void sfresh(int &x)
{
    vfresh(x);
    x = __builtin_amdgcn_readfirstlane(x);
}
template <typename T, int R> __device__ __forceinline__ void refresh(ResCtx<T, R> &c)
{
    vfresh(c.ub);
    vfresh(c.ustep);
    vfresh(c.pxb);
    vfresh(c.pxstep);
    vfresh(c.pzb);
    vfresh(c.pzstep);
    vfresh(c.gb);
    vfresh(c.gstep);
    vfresh(c.own);
    vfresh(c.rbase);
    vfresh(c.dir);
    vfresh(c.col);
    vfresh(c.flags);
    sfresh(c.first);
    sfresh(c.fany);
    sfresh(c.lwb);
    sfresh(c.pxw);
}

// Wait until the border rows that any lane needs (item flags `top`, `bot`) are
// in LDS.  The exchange waves count them in every step, also after a poll
// that ran into its bound, so the wait ends.
template <typename T, int R> __device__ __forceinline__ void wait_borders(const ResCtx<T, R> &c, int top, int bot)
{
    const bool t = __builtin_amdgcn_ballot_w64((c.flags & top) != 0) != 0;
    const bool b = __builtin_amdgcn_ballot_w64((c.flags & bot) != 0) != 0;
    if (!t && !b) return;
    const int *f = reinterpret_cast<const int *>(c.smem + c.flag);
    while ((t && lds_word(f) != c.want_top) || (b && lds_word(f + 1) != c.want_bot)) __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Whether step i of the launch is a strip's last because a poll ran into its
// bound in it: `bad` holds 1 + that step.  A wave may read the word late, when
// an exchange wave is already in the next step and its poll expires there; by
// the number all waves leave after the same step, whose border rows have been
// counted.  One that left a step early would leave the others waiting for its
// count.
__device__ __forceinline__ bool last_step(const int *bad, int i)
{
    const int at = lds_word(bad);
    return at != 0 && at <= i + 1;
}

constexpr bool res_back(int mode) { return mode == 2 || mode == 4; }
constexpr bool res_reads(int mode) { return mode >= 2; }

// A plain thread's step, du_{k+1} and u_{k+1} of its rows.
template <typename T, int R, int MODE, int RM>
__device__ __forceinline__ void plain_a(const ResParams<T> &P, const ResCtx<T, R> &c, Cell<T> (&du)[RM],
                                        const Cell<T> (&c2)[RM], Cell<T> (&ic)[RM], const Cell<T> (&dv)[RM],
                                        int fp, int fmask, bool img, Rsrc dw)
{
    constexpr int V = CellOf<T>::V, HC = ResCtx<T, R>::HC;
    Cell<T> u[RM + 2 * R];
    wait_borders(c, I_BEGIN_TOP, I_BEGIN_BOT);
#pragma unroll
    for (int s = 0; s < 2 * R; ++s)
        if (s >= c.first) u[s] = lds_cell<T>(c.smem, c.ub + (s - R) * c.ustep);
#pragma unroll
    for (int j = 0; j < RM; ++j) {
        // the first row past this thread's own is loaded for row RM - R
        if (j == (RM > R ? RM - R : 0)) wait_borders(c, I_END_TOP, I_END_BOT);
        if (j + 2 * R >= c.first) u[j + 2 * R] = lds_cell<T>(c.smem, c.ub + (j + R) * c.ustep);
        __builtin_amdgcn_sched_barrier(0);
        if (j < c.first) continue;
        const Cell<T> uc = u[j + R];
        T z[V * (2 * HC + 1)];
#pragma unroll
        for (int h = 1; h <= HC; ++h) {
            const Cell<T> a = lds_cell<T>(c.smem, c.ub + j * c.ustep - 16 * h);
            const Cell<T> b = lds_cell<T>(c.smem, c.ub + j * c.ustep + 16 * h);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                z[(HC - h) * V + e] = a.v[e];
                z[(HC + h) * V + e] = b.v[e];
            }
        }
#pragma unroll
        for (int e = 0; e < V; ++e) z[HC * V + e] = uc.v[e];
        Cell<T> f = {};
        if ((c.fany >> j) & 1) {
            if ((fmask >> j) & 1) {
                f = lds_cell<T>(c.smem, fp);
                fp += 16;
            }
        }
        Cell<T> S, un;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const T v = uc.v[e];
            T lx = T(0), lz = T(0);
#pragma unroll
            for (int i = R; i >= 1; --i) {
                lx = fma(P.cx.d2[i], (u[j + R + i].v[e] - v) + (u[j + R - i].v[e] - v), lx);
                lz = fma(P.cz.d2[i], (z[HC * V + e + i] - v) + (z[HC * V + e - i] - v), lz);
            }
            T fe = f.v[e];
            if (MODE == 3) fe += ic[j].v[e] * (-dv[j].v[e]);  // Born source: m1 * (-dWaveOp0_k)
            const T src = fe + (lx + lz);
            S.v[e] = c2[j].v[e] * src;
            du[j].v[e] = fma(P.tc.dt2, S.v[e], du[j].v[e]);
            un.v[e] = v + du[j].v[e];
            if (res_back(MODE) && img) ic[j].v[e] = ic[j].v[e] + v * dv[j].v[e];
        }
        // every lane writes (lanes without rows of their own repeat a
        // neighbour's), but those the wave's first row does not belong to drop it
        int wo = c.ub + j * c.ustep + c.uw, go = c.gb + j * c.gstep;
        if (j == c.first) {
            wo = c.late ? c.drop : wo;
            go = c.late ? kOOB : go;
        }
        lds_put<T>(c.smem, wo, un);
        if (MODE == 1 && img) cell_st<T, true>(dw, go, S);
    }
}

// PML data of a full thread
template <typename T>
struct FullZ {
    static constexpr int V = CellOf<T>::V;
    T szk[V], szm[V], fac[V];
    int zedge;   // bit e: z node e is on the edge of the grid or beyond it
    int sig;     // LDS byte offset of the strip's x profiles {kernel, mesh} per row
    int x0, nx;
    bool exact;
};

// A full thread's step: the PML update of cda2d.hip's march_full.
// XT: the strip has x PML rows or x edges; elsewhere the x profile is zero and
// every row takes the lean form.
template <typename T, int R, int MODE, int RM, bool XT>
__device__ __forceinline__ void full_a(const ResParams<T> &P, const ResCtx<T, R> &c, FullZ<T> &Z,
                                       Cell<T> (&du)[RM], const Cell<T> (&c2)[RM], Cell<T> (&ic)[RM],
                                       const Cell<T> (&dv)[RM], int fp, int fmask, bool img, Rsrc dw)
{
    constexpr int V = CellOf<T>::V, HC = ResCtx<T, R>::HC;
    Cell<T> u[RM + 2 * R];
    const T dt = P.tc.dt, sgn = (c.flags & I_REV) ? T(-1) : T(1);
    wait_borders(c, I_BEGIN_TOP, I_BEGIN_BOT);
#pragma unroll
    for (int s = 0; s < 2 * R; ++s)
        if (s >= c.first) u[s] = lds_cell<T>(c.smem, c.ub + (s - R) * c.ustep);
#pragma unroll
    for (int j = 0; j < RM; ++j) {
        if (j == (RM > R ? RM - R : 0)) wait_borders(c, I_END_TOP, I_END_BOT);
        if (j + 2 * R >= c.first) u[j + 2 * R] = lds_cell<T>(c.smem, c.ub + (j + R) * c.ustep);
        __builtin_amdgcn_sched_barrier(0);
        if (j < c.first) continue;
        T z[V * (2 * HC + 1)], pz[V * (2 * HC + 1)];
#pragma unroll
        for (int h = -HC; h <= HC; ++h) {
            const Cell<T> a = h ? lds_cell<T>(c.smem, c.ub + j * c.ustep + 16 * h) : u[j + R];
            const Cell<T> b = lds_cell<T>(c.smem, c.pzb + j * c.pzstep + 16 * h);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                z[(HC + h) * V + e] = a.v[e];
                pz[(HC + h) * V + e] = b.v[e];
            }
        }
        Cell<T> f = {};
        if ((c.fany >> j) & 1) {
            if ((fmask >> j) & 1) {
                f = lds_cell<T>(c.smem, fp);
                fp += 16;
            }
        }
        T sx = T(0), sxm = T(0);
        bool xedge = false;
        if constexpr (XT) {
            const int row = c.rbase + j * c.dir, x = Z.x0 + row;
            xedge = x == 0 || x == Z.nx - 1;
            // rows a wave marches past its own may lie in the halo: clamped
            const T *sg = reinterpret_cast<const T *>(c.smem + Z.sig) + 2 * clampi(row, 0, c.nr - 1);
            sx = sg[0];
            sxm = sg[1];
        }
        vfresh(Z.zedge);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            vfresh(Z.szk[e]);
            vfresh(Z.szm[e]);
            vfresh(Z.fac[e]);
        }
        const bool lean = !XT || (sx == T(0) && sxm == T(0) && !xedge);
        // Phix along x is read again for every row: a second window would not
        // leave registers for kFullRows rows
        Cell<T> dpxc = {}, dwc, un, pxn, pzn;
#pragma unroll
        for (int i = R; i >= 1; --i) {
            const Cell<T> a = lds_cell<T>(c.smem, c.pxb + (j + i) * c.pxstep);
            const Cell<T> b = lds_cell<T>(c.smem, c.pxb + (j - i) * c.pxstep);
#pragma unroll
            for (int e = 0; e < V; ++e) dpxc.v[e] = fma(P.cx.d1[i - 1], a.v[e] - b.v[e], dpxc.v[e]);
        }
        const Cell<T> pxr = lds_cell<T>(c.smem, c.pxb + j * c.pxstep);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const T v = u[j + R].v[e];
            T lx = T(0), lz = T(0), dux = T(0), duz = T(0), dpz = T(0);
#pragma unroll
            for (int i = R; i >= 1; --i) {
                lx = fma(P.cx.d2[i], (u[j + R + i].v[e] - v) + (u[j + R - i].v[e] - v), lx);
                lz = fma(P.cz.d2[i], (z[HC * V + e + i] - v) + (z[HC * V + e - i] - v), lz);
                dux = fma(P.cx.d1[i - 1], u[j + R + i].v[e] - u[j + R - i].v[e], dux);
                duz = fma(P.cz.d1[i - 1], z[HC * V + e + i] - z[HC * V + e - i], duz);
                dpz = fma(P.cz.d1[i - 1], pz[HC * V + e + i] - pz[HC * V + e - i], dpz);
            }
            // a reversed march took the differences along -x
            dux = dux * sgn;
            const T dpx = dpxc.v[e] * sgn;
            T fe = f.v[e];
            if (MODE == 3) fe += ic[j].v[e] * (-dv[j].v[e]);
            const T src = ((fe + (lx + lz)) + dpx) + dpz;
            const T S = c2[j].v[e] * src;
            const T dm = du[j].v[e];
            const T dni = fma(P.tc.dt2, S, dm);
            const T pxc = pxr.v[e], pzc = pz[HC * V + e];
            const T szk = Z.szk[e], szm = Z.szm[e];
            T dn, dwv, pxv, pzv;
            if (lean) {
                const bool pml = szk != T(0);
                const T dtszk = dt * szk;
                const T pxd = pxc + dtszk * dux;
                const T pzd = (pzc - dtszk * pzc) + (-dtszk) * duz;
                pxv = pml ? pxd : pxc;
                pzv = pml ? pzd : pzc;
                const T szk_dt = szk * P.tc.inv_dt;
                dn = pml ? dm + Z.fac[e] * (S - szk_dt * dm) : dni;
                const T dsz = szm - szk;
                dwv = S + dsz * (dn + dm) * P.tc.inv_2dt;
            } else {
                const bool pml = sx != T(0) || szk != T(0);
                const T pxd = (pxc - dt * sx * pxc) + dt * (szk - sx) * dux;
                const T pzd = (pzc - dt * szk * pzc) + dt * (sx - szk) * duz;
                const T ss = sx + szk, pp = sx * szk;
                const T fac1 = P.tc.two_dt2 / (T(2) + dt * ss);
                pxv = pml ? pxd : pxc;
                pzv = pml ? pzd : pzc;
                dn = pml ? dm + fac1 * ((S - pp * v) - ss * dm * P.tc.inv_dt) : dni;
                dwv = S + ((sxm + szm) - ss) * (dn + dm) * P.tc.inv_2dt + (sxm * szm - pp) * v;
            }
            if (Z.exact) dwv = S;
            const bool edge = xedge || ((Z.zedge >> e) & 1);
            du[j].v[e] = edge ? T(0) : dn;
            un.v[e] = edge ? T(0) : v + dn;
            pxn.v[e] = edge ? T(0) : pxv;
            pzn.v[e] = edge ? T(0) : pzv;
            dwc.v[e] = edge ? T(0) : dwv;
            if (res_back(MODE) && img) ic[j].v[e] = ic[j].v[e] + v * dv[j].v[e];
        }
        int wo = c.ub + j * c.ustep + c.uw, wx = c.pxb + j * c.pxstep + c.pxw2, wz = c.pzb + j * c.pzstep + c.pzw2;
        int go = c.gb + j * c.gstep;
        if (j == c.first) {
            wo = c.late ? c.drop : wo;
            wx = c.late ? c.drop : wx;
            wz = c.late ? c.drop : wz;
            go = c.late ? kOOB : go;
        }
        lds_put<T>(c.smem, wo, un);
        lds_put<T>(c.smem, wx, pxn);
        lds_put<T>(c.smem, wz, pzn);
        if (MODE == 1 && img) cell_st<T, true>(dw, go, dwc);
    }
}

// du, C^2 and the imaging sums (or the Born perturbation) of a thread's rows
template <typename T, int MODE, int RM, typename C>
__device__ __forceinline__ void load_rows(const pysit_amd_batch &B, const pysit_amd_shot &S, const C &c, int x0,
                                          Rsrc rdu, Rsrc ric, Cell<T> (&du)[RM], Cell<T> (&c2)[RM], Cell<T> (&ic)[RM])
{
    constexpr int V = CellOf<T>::V;
    const Rsrc model = make_rsrc(S.model, (long long)(S.mx_hi + 1) * S.mnz * (long long)sizeof(T));
    const Rsrc m1 = make_rsrc(MODE == 3 ? B.born_m1 : S.model,
                              MODE == 3 ? (long long)(S.mx_hi + 1) * S.mnz * (long long)sizeof(T) : 0);
#pragma unroll
    for (int j = 0; j < RM; ++j) {
        // lanes without rows of their own hold a copy of a neighbour's
        const bool own = j > c.first || (j == c.first && !c.late);
        const int go = own ? c.gb + j * c.gstep : kOOB;
        du[j] = cell_ld<T>(rdu, go);
        const int x = x0 + c.rbase + j * c.dir;
        const int mr = clampi(x - S.mx_off, S.mx_lo, S.mx_hi) * S.mnz;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const int z = c.col * V + e;
            const int mo = own && z < S.nz ? (mr + clampi(z - S.mz_off, S.mz_lo, S.mz_hi)) * (int)sizeof(T) : kOOB;
            const T cv = buf_ld<T>(model, mo, 0);
            c2[j].v[e] = cv * cv;
            ic[j].v[e] = MODE == 3 ? buf_ld<T>(m1, mo, 0) : T(0);
        }
        if (res_back(MODE)) ic[j] = cell_ld<T>(ric, go);
    }
}

template <typename T, int RM, typename C>
__device__ __forceinline__ void store_rows(const C &c, Rsrc r, const Cell<T> (&a)[RM])
{
#pragma unroll
    for (int j = 0; j < RM; ++j) cell_st<T>(r, (c.own >> j) & 1 ? c.gb + j * c.gstep : kOOB, a[j]);
}

// The flush of an FP32 window for a strip whose shot takes no step in the
// launch: a window that another run left open (the step kernels, in a segment
// too short for this loop) ends here if one of the launch's slots ends it.
// ic += sums, sums = 0 over the strip's rows, as k_ic_flush does.
__device__ __forceinline__ void flush_idle(const pysit_amd_batch &B, const pysit_amd_shot &S, const int (&d)[kStripInts],
                                           int slot_begin, int slot_end, int window)
{
    if ((slot_begin + window - 1) / window * window >= slot_end) return;
    float *sum = B.ic32 + S.off + (long long)d[1] * S.zs;
    double *ic = B.ic + S.off + (long long)d[1] * S.zs;
    for (int i = threadIdx.x; i < d[2] * S.zs; i += kResThreads) {
        ic[i] += (double)sum[i];
        sum[i] = 0.0f;
    }
}

// the FP32 window's flush: ic += sums, sums = 0
template <int RM, typename C>
__device__ __forceinline__ void flush_rows(const C &c, Rsrc ric, Cell<float> (&ic)[RM])
{
#pragma unroll
    for (int j = 0; j < RM; ++j) {
        if (!((c.own >> j) & 1)) continue;
        const int o = (c.gb + j * c.gstep) * 2;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            Cell<double> d = cell_ld<double>(ric, o + 16 * h);
            d.v[0] += (double)ic[j].v[2 * h];
            d.v[1] += (double)ic[j].v[2 * h + 1];
            cell_st<double>(ric, o + 16 * h, d);
        }
        ic[j] = Cell<float>{};
    }
}

// Phix columns that cross a border: all cells between strips at the x PML, else
// the z PML's.  A border goes in jobs of 64 columns by R rows, those of u
// before those of Phix; none without a neighbour.
__device__ __forceinline__ int border_phix(const int (&d)[kStripInts], int side)
{
    return (d[3] & (side ? S_PXBOT : S_PXTOP)) ? d[21] : d[6] + d[7];
}
__device__ __forceinline__ int border_jobs(const int (&d)[kStripInts], int side)
{
    return d[19 + side] >= 0 ? (d[21] + 63) / 64 + (border_phix(d, side) + 63) / 64 : 0;
}

// Whether the step of k is imaged.
__device__ __forceinline__ bool res_imaged(const pysit_amd_batch &B, int k)
{
    return B.dw && (B.imaging_period == 1 || k % B.imaging_period == 0);
}

// The steps of one strip by its computing waves of one kind (1 plain, 2
// full, 3 full with x PML rows).
template <typename T, int R, int MODE, int KIND>
__device__ __forceinline__ void strip_loop(const pysit_amd_batch &B, const ResParams<T> &P, const pysit_amd_shot &S,
                                           const int (&d)[kStripInts], ResCtx<T, R> &c, int first_slot, int n)
{
    constexpr int V = CellOf<T>::V, SZ = sizeof(T);
    constexpr int RM = KIND != 1 ? kFullRows : kPlainRows;
    const long long nb = (long long)S.nx * S.zs * SZ;
    const int kshift = __builtin_amdgcn_readfirstlane(S.kshift);
    const int k0 = first_slot - kshift;
    const int cur = (res_back(MODE) ? S.nt - 1 - k0 : k0) & 1, fin = (cur + n) & 1;
    const Rsrc rdu = make_rsrc((T *)B.du + S.off, nb);
    const Rsrc ru = make_rsrc((const T *)B.u[cur] + S.off, nb);
    // imaging sums between launches: the FP32 window's buffer or the FP64 one
    const Rsrc ric = make_rsrc(MODE == 4 ? (const void *)(B.ic32 + S.off)
                                         : (MODE == 2 ? (const void *)(B.ic + S.off) : B.u[0]),
                               res_back(MODE) ? nb : 0);
    const Rsrc ric64 = make_rsrc(MODE == 4 ? (const void *)(B.ic + S.off) : B.u[0], MODE == 4 ? nb * 2 : 0);
    const int x0 = d[1];

    Cell<T> du[RM], c2[RM], ic[RM], dv[RM];
    FullZ<T> Z;
    load_rows<T, MODE, RM>(B, S, c, x0, rdu, ric, du, c2, ic);
#pragma unroll
    for (int j = 0; j < RM; ++j)
        if ((c.own >> j) & 1) lds_put<T>(c.smem, c.ub + j * c.ustep, cell_ld<T>(ru, c.gb + j * c.gstep));
    if constexpr (KIND != 1) {
        const Rsrc rpx = make_rsrc((const T *)B.phix[cur] + S.off, nb);
        const Rsrc rpz = make_rsrc((const T *)B.phiz[cur] + S.off, nb);
#pragma unroll
        for (int j = 0; j < RM; ++j)
            if ((c.own >> j) & 1) {
                const int go = c.gb + j * c.gstep;
                lds_put<T>(c.smem, c.pxb + j * c.pxstep, cell_ld<T>(rpx, go));
                lds_put<T>(c.smem, c.pzb + j * c.pzstep, cell_ld<T>(rpz, go));
            }
        Z.zedge = 0;
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const int z = c.col * V + e;
            const bool in = z < S.nz;
            Z.szk[e] = in ? sigma_kernel<T>((const T *)S.zl, S.nzl, (const T *)S.zr, S.nzr, z, S.nz) : T(0);
            Z.szm[e] = in ? sigma_mesh<T>((const T *)S.zl, S.nzl, (const T *)S.zr, S.nzr, z, S.nz) : T(0);
            Z.fac[e] = P.tc.two_dt2 / (T(2) + P.tc.dt * Z.szk[e]);
            Z.zedge |= (z == 0 || z >= S.nz - 1) ? 1 << e : 0;
        }
        Z.sig = d[17];
        Z.x0 = x0;
        Z.nx = S.nx;
        Z.exact = B.dw_form == 1;
    }
    const int fblk = P.adjoint_tables ? d[30] : d[29];
    const int2 fi = P.n_inj && fblk >= 0 ? P.finfo[(long long)fblk * kResThreads +
                                                             (P.items[d[28] * kResThreads + threadIdx.x].w >> 16)] : make_int2(0, 0);
    const int fp = d[16] + fi.x * 16;
    c.fany = 0;
    for (int j = 0; j < RM; ++j) c.fany |= __builtin_amdgcn_ballot_w64((fi.y >> j) & 1) ? 1 << j : 0;
    int f_at = fp;
    const bool dw_on = MODE >= 1 && B.dw;
    const T *dw_base = dw_on ? (const T *)B.dw + S.off : (const T *)B.u[0];
    auto dw_rsrc = [&](int slot, bool on) {
        on = on && dw_on;
        return make_rsrc(dw_base + (on ? (long long)(slot - P.seg_base) * B.total_n : 0), on ? nb : 0);
    };
    // The history values of a step are loaded together once the march before
    // it has used its own: they arrive while the wave waits at the barrier and
    // for the border rows.  Loaded row by row within the march, every row
    // waited for the load before it (loads return in order): 2.3 times the
    // time per row.
    auto load_dw = [&](int slot, bool on) {
        const Rsrc r = dw_rsrc(slot, on);
#pragma unroll
        for (int j = 0; j < RM; ++j)
            dv[j] = cell_ld<T, true>(r, j > c.first || (j == c.first && !c.late) ? c.gb + j * c.gstep : kOOB);
    };
    if constexpr (res_reads(MODE)) load_dw(first_slot, true);
    lds_sync();

    const int jobs_top = border_jobs(d, 0), jobs_bot = border_jobs(d, 1);
    bool bad = lds_word(reinterpret_cast<const int *>(c.smem + c.flag + 12)) != 0;
    for (int i = 0; i < n && !bad; ++i) {
        const int slot = first_slot + i * P.direction, k = slot - kshift;
        const bool more = i + 1 < n;
        const bool img = res_imaged(B, k);
        const bool next = res_reads(MODE) && more && res_imaged(B, k + P.direction);
        c.want_top = jobs_top * (i + 1);
        c.want_bot = jobs_bot * (i + 1);
        {
            refresh(c);
            int fmask = fi.y;
            vfresh(fmask);
            const Rsrc dw = dw_rsrc(slot, true);
            if constexpr (KIND == 1) plain_a<T, R, MODE, RM>(P, c, du, c2, ic, dv, f_at, fmask, img, dw);
            else full_a<T, R, MODE, RM, KIND == 3>(P, c, Z, du, c2, ic, dv, f_at, fmask, img, dw);
        }
        if constexpr (MODE == 4) {
            // a shot that starts inside a window has its last sums after step 0
            if (window_end(slot, P.direction, P.window) || k == 0) flush_rows<RM>(c, ric64, ic);
        }
        if constexpr (res_reads(MODE)) load_dw(more ? slot + P.direction : slot, next);
        // the next step reads the other copy
        c.ub += c.uw;
        c.pxb += c.pxw2;
        c.pzb += c.pzw2;
        c.uw = -c.uw;
        c.pxw2 = -c.pxw2;
        c.pzw2 = -c.pzw2;
        f_at = fp + ((i + 1) & 1) * d[27];
        lds_sync();
        bad = last_step(reinterpret_cast<const int *>(c.smem + c.flag + 8), i);
    }
    // state back to memory; after a poll that ran into its bound, NaN
    const Rsrc wu = make_rsrc((T *)B.u[fin] + S.off, nb);
    const T poison = bad ? __builtin_nan("") : T(0);
#pragma unroll
    for (int j = 0; j < RM; ++j) {
        if (!((c.own >> j) & 1)) continue;
        Cell<T> u = lds_cell<T>(c.smem, c.ub + j * c.ustep);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            if (bad) u.v[e] = poison;
            if (bad) ic[j].v[e] = poison;
        }
        cell_st<T>(wu, c.gb + j * c.gstep, u);
    }
    store_rows<T, RM>(c, rdu, du);
    if (res_back(MODE)) store_rows<T, RM>(c, ric, ic);
    if constexpr (KIND != 1) {
        const Rsrc wpx = make_rsrc((T *)B.phix[fin] + S.off, nb);
        const Rsrc wpz = make_rsrc((T *)B.phiz[fin] + S.off, nb);
#pragma unroll
        for (int j = 0; j < RM; ++j)
            if ((c.own >> j) & 1) {
                cell_st<T>(wpx, c.gb + j * c.gstep, lds_cell<T>(c.smem, c.pxb + j * c.pxstep));
                cell_st<T>(wpz, c.gb + j * c.gstep, lds_cell<T>(c.smem, c.pzb + j * c.pzstep));
            }
    }
}

// ---- exchange waves -------------------------------------------------------------
// d[23] waves of a strip; wave `me` takes every d[23]-th job of the two
// borders, at most kJobs of them (the host sees to it), and its share of the
// receivers' nodes and sources.  The code is kept short: one wave of eight
// runs it, and once the loops of a strip's waves outgrow the instruction
// cache, this one waits for its own instructions (the 14 stores of 36 rows of
// 341 nodes took 9000 cycles unrolled over 16 packed operations).
constexpr int kJobs = 6;
constexpr int kMine = 8;        // sources and receiver nodes per lane kept in registers
constexpr int kXchgTags = 64;   // tags per side of a strip
constexpr int kAgent = 16;      // buffer access past the caches of the XCD (sc1)

__device__ __forceinline__ unsigned *border_tags(char *xchg, long long stride, int strip, int side)
{
    return reinterpret_cast<unsigned *>(xchg + strip * stride) + side * kXchgTags;
}
__device__ __forceinline__ char *border_data(char *xchg, long long stride, int strip, int side, int par, int cells)
{
    return xchg + strip * stride + 2 * kXchgTags * 4 + (long long)((side * 2 + par) * cells) * 16;
}

template <typename T, int R, int MODE>
__device__ __forceinline__ void exchange_loop(const ResParams<T> &P, const int (&d)[kStripInts], char *smem, int lwb,
                                              int pxw, int flag, int me, int first_slot, int n)
{
    constexpr int SZ = sizeof(T), HC = ResCtx<T, R>::HC;
    int *f = reinterpret_cast<int *>(smem + flag);
    int *bad = f + 2;
    if (me >= d[23]) {  // an idle wave keeps the others company at the barriers
        lds_sync();
        if (lds_word(bad + 1)) return;
        for (int i = 0; i < n; ++i) {
            lds_sync();
            if (last_step(bad, i)) break;
        }
        return;
    }
    const int waves = d[23], lanes = waves * 64, lane = threadIdx.x & 63, lid = me * 64 + lane;
    const int jobs0 = border_jobs(d, 0), jobs = jobs0 + border_jobs(d, 1);
    // how many are this wave's, on both sides and at the top
    const int mine = jobs > me ? (jobs - me + waves - 1) / waves : 0;
    const int mine0 = jobs0 > me ? (jobs0 - me + waves - 1) / waves : 0;
    // per job: LDS cell of this lane's column in the first row to publish, from
    // there to the first row to fill, bytes per row and per copy, offset of the
    // column in the border's data (out of range past the columns)
    int src[kJobs], fill[kJobs], rowb[kJobs], copy[kJobs], off[kJobs], at[kJobs];
#pragma unroll
    for (int m = 0; m < kJobs; ++m) {
        const int job = me + m * waves, side = job >= jobs0, k = job - (side ? jobs0 : 0);
        const int nzc = d[21], fl = d[4], fr = d[5], nu = (nzc + 63) / 64, px = border_phix(d, side);
        const bool phi = k >= nu;
        const int q = (phi ? k - nu : k) * 64 + lane;
        const bool live = m < mine && q < (phi ? px : nzc);
        // Phix column q: cell q, or cell of the z band
        const int cell = px == nzc || q < d[6] ? q : nzc - d[7] + (q - d[6]);
        rowb[m] = phi ? pxw : lwb;
        copy[m] = phi ? d[25] : d[24];
        src[m] = (side ? d[2] : R) * rowb[m] +
                 (phi ? d[14] + (cell < fl ? cell : cell - (nzc - fr) + fl) * 16 : (HC + q) * 16);
        fill[m] = side ? R * rowb[m] : -R * rowb[m];
        src[m] = live ? src[m] : 0;
        off[m] = live ? lane * 16 : kOOB;
        at[m] = __builtin_amdgcn_readfirstlane(k * R * 1024);
    }
    // lane m of the wave watches over job m's tag
    const int my_job = me + lane * waves, my_side = my_job >= jobs0;
    const bool tagged = lane < mine;
    const int tag_at = my_job - (my_side ? jobs0 : 0);
    unsigned *put = border_tags(P.xchg, P.xstride, d[22], my_side) + tag_at;
    const unsigned *get = border_tags(P.xchg, P.xstride, tagged ? (my_side ? d[20] : d[19]) : 0, 1 - my_side) + tag_at;
    const int inj0 = P.adjoint_tables ? d[12] : d[10], inj1 = P.n_inj ? (P.adjoint_tables ? d[13] : d[11]) : inj0;
    const int rec0 = d[8], rec1 = P.record ? d[9] : rec0;
    int il[kMine], rl[kMine];
    T fv[kMine];
#pragma unroll
    for (int q = 0; q < kMine; ++q) {
        const int i = inj0 + lid + q * lanes, r = rec0 + lid + q * lanes;
        il[q] = i < inj1 ? d[16] + P.inj_lds[i] * SZ : -1;
        rl[q] = r < rec1 ? P.rec_lds[r] : -1;
    }
    for (int i = inj0 + lid; i < inj1; i += lanes)
        *reinterpret_cast<T *>(smem + d[16] + P.inj_lds[i] * SZ) =
            P.pre[(long long)(first_slot - P.slot_begin) * P.n_inj + i];
    lds_sync();
    if (lds_word(bad + 1)) return;
    for (int i = 0; i < n; ++i) {
        const int slot = first_slot + i * P.direction;
        const bool more = i + 1 < n;
        const unsigned tag = P.epoch + 1 + i;
        const int par = i & 1, bytes = P.xcells * 16;
        u32x4 v[kJobs][R];
        if (mine) {
            const Rsrc top = make_rsrc(border_data(P.xchg, P.xstride, d[22], 0, par, P.xcells), bytes);
            const Rsrc bot = make_rsrc(border_data(P.xchg, P.xstride, d[22], 1, par, P.xcells), bytes);
#pragma unroll
            for (int m = 0; m < kJobs; ++m)
                if (m < mine) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        v[m][r] = *reinterpret_cast<const u32x4 *>(smem + src[m] + par * copy[m] + r * rowb[m]);
                }
#pragma unroll
            for (int m = 0; m < kJobs; ++m)
                if (m < mine) {
                    const Rsrc to = m < mine0 ? top : bot;
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        __builtin_amdgcn_raw_buffer_store_b128(v[m][r], to, off[m], at[m] + r * 1024, kAgent);
                }
            // the cells are where every reader sees them before their tags are
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_s_waitcnt(0);
            if (tagged) __hip_atomic_store(put, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // the next step's source values, on their way while this step runs
        const T *pn = P.pre + (long long)(slot + P.direction - P.slot_begin) * P.n_inj + inj0;
        if (more && inj1 > inj0) {
#pragma unroll
            for (int q = 0; q < kMine; ++q)
                if (il[q] >= 0) fv[q] = pn[lid + q * lanes];
        }
        if (mine) {
            int spins = 0;
            // the neighbour may be a step ahead: its other buffer holds this one
            while (tagged && (int)(__hip_atomic_load(get, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - tag) < 0)
                if (++spins > P.spin) {
                    __hip_atomic_store(bad, i + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    break;
                }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            const Rsrc top = make_rsrc(border_data(P.xchg, P.xstride, jobs0 ? d[19] : d[22], 1, par, P.xcells), bytes);
            const Rsrc bot = make_rsrc(border_data(P.xchg, P.xstride, jobs > jobs0 ? d[20] : d[22], 0, par, P.xcells),
                                       bytes);
#pragma unroll
            for (int m = 0; m < kJobs; ++m)
                if (m < mine) {
                    const Rsrc from = m < mine0 ? top : bot;
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        v[m][r] = __builtin_amdgcn_raw_buffer_load_b128(from, off[m], at[m] + r * 1024, kAgent);
                }
#pragma unroll
            for (int m = 0; m < kJobs; ++m)
                if (m < mine && off[m] != kOOB) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        *reinterpret_cast<u32x4 *>(smem + src[m] + fill[m] + par * copy[m] + r * rowb[m]) = v[m][r];
                }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            const int done = lane ? mine - mine0 : mine0;
            if (lane < 2 && done)
                __hip_atomic_fetch_add(f + lane, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        // receivers read u_k
        if (rec1 > rec0) {
            T *rb = P.recbuf + (long long)(slot - P.slot_begin) * P.n_rec + rec0;
#pragma unroll
            for (int q = 0; q < kMine; ++q)
                if (rl[q] >= 0) rb[lid + q * lanes] = *reinterpret_cast<const T *>(smem + rl[q] + par * d[24]);
            for (int r = rec0 + lid + kMine * lanes; r < rec1; r += lanes)
                rb[r - rec0] = *reinterpret_cast<const T *>(smem + P.rec_lds[r] + par * d[24]);
        }
        if (more && inj1 > inj0) {
            const int fn = (1 - par) * d[27];
#pragma unroll
            for (int q = 0; q < kMine; ++q)
                if (il[q] >= 0) *reinterpret_cast<T *>(smem + il[q] + fn) = fv[q];
            for (int q = inj0 + lid + kMine * lanes; q < inj1; q += lanes)
                *reinterpret_cast<T *>(smem + d[16] + P.inj_lds[q] * SZ + fn) = pn[q - inj0];
        }
        lds_sync();
        if (last_step(bad, i)) {
            if (lane == 0) {
                __hip_atomic_store(P.stop, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(P.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
            break;
        }
    }
}

template <typename T, int R, int MODE>
__global__ __launch_bounds__(kResThreads) void k_resident2d(const pysit_amd_batch B, const ResParams<T> P)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x;
    const int strip = P.strip0 + xcd_block(blockIdx.x, gridDim.x);
    // the strip's numbers as scalars: read from memory inside the loop they
    // would wait for the stores in flight
    int d[kStripInts];
#pragma unroll
    for (int i = 0; i < kStripInts; ++i)
        d[i] = __builtin_amdgcn_readfirstlane(P.strips[(long long)strip * kStripInts + i]);
    const pysit_amd_shot &S = B.shots[d[0]];
    const int kshift = __builtin_amdgcn_readfirstlane(S.kshift);
    constexpr int SZ = sizeof(T), HC = ResCtx<T, R>::HC;
    // this shot's steps of the launch
    const int lo = max(P.slot_begin, kshift), end = P.slot_begin + P.n_steps;
    const int n = end - lo;
    const int first_slot = P.direction > 0 ? lo : end - 1;
    // receivers of a shot that starts inside the launch: its earlier slots
    // hold no values and are not read
    if (n <= 0) {
        if constexpr (MODE == 4) flush_idle(B, S, d, P.slot_begin, end, P.window);
        return;
    }

    for (int i = tid; i < d[18] / 16 + 2; i += kResThreads)
        *reinterpret_cast<u32x4 *>(smem + 16 * i) = u32x4{0, 0, 0, 0};
    lds_sync();
    // one read for all waves, which look at it after their first barrier
    if (tid == 0)
        *reinterpret_cast<int *>(smem + d[18] + 12) =
            __hip_atomic_load(P.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    {
        // x profiles of the strip's rows
        T *sg = reinterpret_cast<T *>(smem + d[17]);
        for (int r = tid; r < d[2]; r += kResThreads) {
            const int x = d[1] + r;
            sg[2 * r] = sigma_kernel<T>((const T *)S.xl, S.nxl, (const T *)S.xr, S.nxr, x, S.nx);
            sg[2 * r + 1] = sigma_mesh<T>((const T *)S.xl, S.nxl, (const T *)S.xr, S.nxr, x, S.nx);
        }
    }
    const int4 it = P.items[d[28] * kResThreads + tid];
    const int kind = __builtin_amdgcn_readfirstlane((it.y / I_KIND) & 3);
    const int nzc = d[21], fl = d[4], fr = d[5];
    // a row's zero cells at the right are the next row's at the left
    const int lwb = (nzc + HC) * 16, pxw = (fl + fr) * 16, pzw = (fl + fr + 2 * HC) * 16;
    if (kind == 3) {
        exchange_loop<T, R, MODE>(P, d, smem, lwb, pxw, d[18], __builtin_amdgcn_readfirstlane(it.x), first_slot, n);
        return;
    }
    ResCtx<T, R> c;
    c.smem = smem;
    c.flag = d[18];
    c.drop = d[18] + 16;
    c.rbase = it.x;
    c.flags = it.y;
    c.own = it.z & 0xffff;
    c.first = __builtin_amdgcn_readfirstlane((it.z >> 16) & 0xff);
    c.late = (it.z >> 24) & 1;
    c.col = it.w & 0xffff;
    c.dir = (it.y & I_REV) ? -1 : 1;
    c.nr = d[2];
    c.lwb = lwb;
    c.pxw = pxw;
    c.ub = (R + c.rbase) * lwb + (HC + c.col) * 16;
    c.ustep = c.dir * lwb;
    const int fc = c.col < fl ? c.col : c.col - (nzc - fr) + fl;
    c.pxb = d[14] + (R + c.rbase) * pxw + fc * 16;
    c.pxstep = c.dir * pxw;
    c.pzb = d[15] + c.rbase * pzw + (HC + fc + (c.col < fl ? 0 : HC)) * 16;
    c.pzstep = c.dir * pzw;
    c.uw = d[24];
    c.pxw2 = d[25];
    c.pzw2 = d[26];
    c.gb = (d[1] + c.rbase) * S.zs * SZ + c.col * 16;
    c.gstep = c.dir * S.zs * SZ;
    if (kind == 2 && (d[3] & S_XTYPE)) strip_loop<T, R, MODE, 3>(B, P, S, d, c, first_slot, n);
    else if (kind == 2) strip_loop<T, R, MODE, 2>(B, P, S, d, c, first_slot, n);
    else strip_loop<T, R, MODE, 1>(B, P, S, d, c, first_slot, n);
}

// ---- receivers ---------------------------------------------------------------
// Traces from the receiver nodes' values of a run of slots: 16 lanes per
// receiver and kRecSlots slots, each lane's entries and the final butterfly
// in the step loop's order (rec_gather, sample_group), so the sums are the
// same.  An entry's node and weight are loaded once for all slots.
constexpr int kRecSlots = 8;
template <typename T>
__global__ __launch_bounds__(256) void k_rec_sum(const pysit_amd_batch B, const int *__restrict__ node,
                                                 const T *__restrict__ recbuf, int n_rec, int slot_begin, int n_slots)
{
    const int rec = blockIdx.x * 16 + (threadIdx.x >> 4), g = threadIdx.x & 15;
    const int s0 = blockIdx.y * kRecSlots;
    const bool act = rec < B.n_rec;
    int4 rd = make_int4(0, 0, 0, 0);
    if (act) rd = reinterpret_cast<const int4 *>(B.recs)[rec];
    double acc[kRecSlots];
    const T *row[kRecSlots];
#pragma unroll
    for (int q = 0; q < kRecSlots; ++q) {
        acc[q] = 0.0;
        row[q] = recbuf + (long long)min(s0 + q, n_slots - 1) * n_rec;
    }
    for (int e = rd.z + g; e < rd.w; e += 16) {
        const int m = node[e];
        const double w = B.rec_w[e];
#pragma unroll
        for (int q = 0; q < kRecSlots; ++q) acc[q] = __builtin_fma(w, (double)row[q][m], acc[q]);
    }
#pragma unroll
    for (int q = 0; q < kRecSlots; ++q) {
#pragma unroll
        for (int m = 8; m >= 1; m >>= 1) acc[q] += __shfl_xor(acc[q], m, 16);
    }
    if (act && g == 0) {
        const pysit_amd_shot &S = B.shots[rd.x];
#pragma unroll
        for (int q = 0; q < kRecSlots; ++q) {
            const int k = slot_begin + s0 + q - S.kshift;
            if (s0 + q < n_slots && k >= 0 && k < S.nt) S.trace[(long long)k * S.nrec + rd.y] = acc[q];
        }
    }
}

// NaN into the traces and the image of a batch whose wait expired.  Queued
// behind every forward and every adjoint: 256 workgroups that read one word.
__global__ __launch_bounds__(256) void k_res_seal(const pysit_amd_batch B, const int *stop)
{
    if (!*stop) return;
    const long long at = (long long)blockIdx.x * 256 + threadIdx.x, step = (long long)gridDim.x * 256;
    if (B.ic)
        for (long long i = at; i < B.total_n; i += step) B.ic[i] = __builtin_nan("");
    if (!B.n_rec) return;
    for (int s = 0; s < B.n_shots; ++s) {
        const pysit_amd_shot &S = B.shots[s];
        for (long long i = at; i < (long long)S.nt * S.nrec; i += step) S.trace[i] = __builtin_nan("");
    }
}

// ---- host ---------------------------------------------------------------------
int resident_seal(const pysit_amd_batch &B, const int *stop, hipStream_t st)
{
    hipLaunchKernelGGL(k_res_seal, dim3(256), dim3(256), 0, st, B, stop);
    PA_HIP(hipGetLastError());
    return PYSIT_AMD_OK;
}

int inj_precompute(const pysit_amd_batch &B, int slot_begin, int slot_end, int seg_base, hipStream_t st);

template <typename T, int R, int MODE>
static int launch_res(const pysit_amd_batch &B, const ResParams<T> &P, int blocks, int lds, hipStream_t st)
{
    auto k = k_resident2d<T, R, MODE>;
    PA_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    void *args[] = {(void *)&B, (void *)&P};
    PA_HIP(hipLaunchCooperativeKernel((const void *)k, dim3(blocks), dim3(kResThreads), args, lds, st));
    return PYSIT_AMD_OK;
}

template <typename T, int R>
static int launch_res_mode(int kmode, const pysit_amd_batch &B, const ResParams<T> &P, int blocks, int lds,
                           hipStream_t st)
{
    switch (kmode) {
    case 0: return launch_res<T, R, 0>(B, P, blocks, lds, st);
    case 1: return launch_res<T, R, 1>(B, P, blocks, lds, st);
    case 2:
        if constexpr (sizeof(T) == 8) return launch_res<T, R, 2>(B, P, blocks, lds, st);
        break;
    case 3: return launch_res<T, R, 3>(B, P, blocks, lds, st);
    case 4:
        if constexpr (sizeof(T) == 4) return launch_res<T, R, 4>(B, P, blocks, lds, st);
        break;
    }
    set_error("the resident loop has no such mode");
    return PYSIT_AMD_EINVAL;
}

template <typename T>
static int launch_res_r(int r, int kmode, const pysit_amd_batch &B, const ResParams<T> &P, int blocks, int lds,
                        hipStream_t st)
{
    switch (r) {
    case 1: return launch_res_mode<T, 1>(kmode, B, P, blocks, lds, st);
    case 2: return launch_res_mode<T, 2>(kmode, B, P, blocks, lds, st);
    case 3: return launch_res_mode<T, 3>(kmode, B, P, blocks, lds, st);
    case 4: return launch_res_mode<T, 4>(kmode, B, P, blocks, lds, st);
    }
    set_error("order must be 2, 4, 6 or 8");
    return PYSIT_AMD_EINVAL;
}

template <typename T>
int run2d_resident(const pysit_amd_batch &B, const pysit_amd_resident &Q, int mode, int slot_begin, int slot_end,
                   int direction, int seg_base, int record, hipStream_t st)
{
    const int r = B.order / 2;
    const bool window = mode == 2 && B.ic32 != nullptr;
    const int kmode = window ? 4 : mode;
    PA_CHECK(mode != 2 || (sizeof(T) == 8 ? !window : window),
             "the resident adjoint sums an FP32 batch in the FP32 window, an FP64 batch in FP64");
    PA_CHECK(mode != 2 || B.dw, "the resident adjoint images every run (dw must be given)");
    ResParams<T> P{};
    P.cx = axis_coef<T>(r, B.dx);
    P.cz = axis_coef<T>(r, B.dz);
    P.tc = time_coef<T>(B.dt);
    const int adj = mode == 2;
    P.adjoint_tables = adj;
    P.strips = Q.strips;
    P.items = (const int4 *)Q.items;
    P.finfo = (const int2 *)Q.finfo[adj];
    P.inj_lds = Q.inj_lds[adj];
    P.rec_lds = Q.rec_lds;
    P.pre = (const T *)Q.pre;
    P.recbuf = (T *)Q.recbuf;
    P.xchg = (char *)Q.xchg;
    P.xstride = Q.xchg_stride;
    P.xcells = Q.xchg_cells;
    P.err = Q.err;
    P.stop = Q.stop;
    P.direction = direction;
    P.seg_base = seg_base;
    P.n_inj = mode == 3 ? 0 : Q.n_inj[adj];
    P.n_rec = Q.n_rec_nodes;
    P.record = record && mode != 2 && Q.n_rec_nodes > 0;
    P.window = window ? B.ic_window : 0;
    P.spin = Q.spin;
    // source values and receiver nodes are kept for a chunk of slots at a time
    int chunk = slot_end - slot_begin;
    if (P.n_inj) chunk = std::min(chunk, Q.pre_slots);
    if (P.record) chunk = std::min(chunk, Q.rec_slots);
    PA_CHECK(chunk >= 1, "the resident loop's buffers hold no slot");
    pysit_amd_batch I = B;  // the source tables in strip order, for k_inj_pre
    I.inj_nptr = Q.inj_nptr[adj];
    I.inj_chan = Q.inj_chan[adj];
    I.inj_w = Q.inj_w[adj];
    I.inj_node_shot = Q.inj_shot[adj];
    I.n_inj_nodes = P.n_inj;
    I.inj_pre = Q.pre;
    for (int done = 0; done < slot_end - slot_begin;) {
        const int len = std::min(chunk, slot_end - slot_begin - done);
        const int j0 = direction > 0 ? slot_begin + done : slot_end - done - len;
        if (P.n_inj) {
            const int rc = inj_precompute(I, j0, j0 + len, j0, st);
            if (rc) return rc;
        }
        P.slot_begin = j0;
        P.n_steps = len;
        if (*Q.epoch > 0xffffffffu - (unsigned)len - 8u) {
            set_error("the resident loop's step tags ran out: clear its exchange buffer");
            return PYSIT_AMD_EINVAL;
        }
        P.epoch = *Q.epoch;
        for (int g = 0; g < Q.n_groups; ++g) {
            P.strip0 = Q.group_begin[g];
            const int rc = launch_res_r<T>(r, kmode, B, P, Q.group_begin[g + 1] - Q.group_begin[g], Q.group_lds[g], st);
            if (rc) return rc;
        }
        *Q.epoch += (unsigned)len + 2u;
        if (P.record) {
            hipLaunchKernelGGL(k_rec_sum<T>, dim3((unsigned)((B.n_rec + 15) / 16), (unsigned)((len + kRecSlots - 1) / kRecSlots)),
                               dim3(256), 0, st, B, Q.rec_node, (const T *)Q.recbuf, Q.n_rec_nodes, j0, len);
            PA_HIP(hipGetLastError());
        }
        done += len;
    }
    return PYSIT_AMD_OK;
}

template int run2d_resident<float>(const pysit_amd_batch &, const pysit_amd_resident &, int, int, int, int, int, int,
                                   hipStream_t);
template int run2d_resident<double>(const pysit_amd_batch &, const pysit_amd_resident &, int, int, int, int, int, int,
                                    hipStream_t);

// rows of a thread's column, plain and PML; what an exchange wave takes
void resident_rows(int *plain, int *full, int *threads, int *jobs, int *tags)
{
    *jobs = kJobs;
    *tags = kXchgTags;
    *plain = kPlainRows;
    *full = kFullRows;
    *threads = kResThreads;
}

}  // namespace pa
