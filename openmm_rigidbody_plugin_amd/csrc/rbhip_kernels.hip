// Hot-path kernels of the rigid-body step for gfx950 (wave64).
//
//   k_part1  integratePart1 (reference openmmapi/src/RigidBodySystem.cpp:170-187):
//            free atoms: v += F/m dt/2, r += v dt; bodies: r_cm += p_cm dt/M
//            (FP64), free rotation (NO-SQUISH with an FP64-accurate composite
//            rotation, or the FP64 exact solution), FP64 renormalisation of q,
//            atom positions r_j = r_cm + A(q)^T d_j.
//   k_part2  integratePart2 (RigidBodySystem.cpp:193-204): free atoms
//            v += F/m dt/2; bodies: F = sum f_j, tau = sum delta_j x f_j (FP64),
//            half-kick of p_cm and L, atom velocities v_cm + w_s x delta_j,
//            FP64 kinetic-energy partials per tile, then the next step's first
//            half-kick (the reference applies it at the start of part1 with the
//            same F and torque, so folding it here is the same arithmetic).
//   k_fused  part2 of step n + part1 of step n+1 in one pass (interior steps
//            of RigidBodyIntegrator::step(k)).
//   k_steps  several steps of systems whose atoms' forces depend on no other
//            atom: part 1, then [forces, k_fused] boundaries, in registers.
//   k_forces the force-field slot: harmonic tethers and harmonic bonds.
//
// Body state per body: q (Real4), body-frame L and p_cm (3 Reals each), iI =
// (1/I, 1/M), r_cm (FP64).  The reference's quaternion momentum is
// pi = 2 B(q) L, its torque kick pi += C(q) tau dt is L += A(q) tau dt / 2.
// Every workgroup walks the tile list with a grid stride, so one launch
// covers any number of systems (the batch path) and any grid cap.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "rbhip_access.h"
#include "rbhip_kernels.h"

namespace rbhip {

__device__ __forceinline__ int lane_shift(int lanes) { return __ffs(lanes) - 1; }

// ---------------------------------------------------------------------------
// block reduction of up to 4 doubles per lane into slot `slot` of `out`
// (fixed order: wave shuffles, then waves in index order)
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

template <int NV>
__device__ void block_reduce_store(double (&v)[NV], double* out, int slot) {
    __shared__ double red[8][4];
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int c = 0; c < NV; c++) {
        double s = wave_sum(v[c]);
        if (lane == 0) red[wave][c] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int nw = (blockDim.x + 63) >> 6;
        for (int c = 0; c < NV; c++) {
            double s = 0.0;
            for (int w = 0; w < nw; w++) s += red[w][c];
            out[4 * (size_t)slot + c] = s;
        }
    }
    __syncthreads();
}

__device__ __forceinline__ double xor_sum(double v, int lanes) {
    for (int m = 1; m < lanes; m <<= 1) v += __shfl_xor(v, m, 64);
    return v;
}

// ---------------------------------------------------------------------------
// body state and the per-atom loops
// ---------------------------------------------------------------------------
template <class Real> struct Body {
    Q4<Real> q;
    V3<Real> L, p, invI;
    Real invM;
};

// body k's state, with 1/I and 1/M read at body ks (the body whose inertia it
// shares, or itself)
template <class Real> __device__ __forceinline__ Body<Real> load_body(const DevSys& S, int k, int ks) {
    Q4<Real> iI = ld4<Real>(S.iI, ks);
    return Body<Real>{ld4<Real>(S.q, k), ldp3<Real>(S.L, k), ldp3<Real>(S.pcm, k), V3<Real>{iI.a, iI.b, iI.c}, iI.d};
}

// atoms per lane a strided per-body loop loads before it uses any (bodies of
// more than 6 atoms, several lanes each)
constexpr int STRIDED_BATCH = 8;

// Adopted arrays lie in their caller's order, so a wave's accesses to them are
// scattered, and a loop over a lane's atoms waits for a round trip per atom,
// behind the stores of the atom before (which may alias).  So a lane loads
// several atoms before it stores any.  How many, for the atoms' forces: 4 in
// mixed precision (100k waters 10.5 -> 9.1 us), 2 in double (40k waters 6.6 ->
// 6.2; 4: 6.9).  For free atoms in the step kernels: 4 in mixed precision
// (300k free atoms, part 1 41.2 -> 37.4 us), 1 in double, where the registers
// of 4 cost bodies in the same launch more (20k mixed bodies and 30k free
// atoms, exact, part 1: 8.8 us, with 4 9.3; 300k free atoms 32.2, with 4
// 29.9).  The library's own arrays, whose accesses are coalesced, gain nothing
// from a batch.
template <class Real, class IO> constexpr int force_batch() { return !IO::adopted ? 1 : sizeof(Real) == 4 ? 4 : 2; }
template <class Real, class IO> constexpr int free_batch() { return IO::adopted && sizeof(Real) == 4 ? 4 : 1; }

// A(q)^T d of atom u of a lane's batch.  (The first of a batch rounds its y
// product and the others their x product, as the compiler fused them when
// these loops were tuned; one rule for all kernels keeps their trajectories
// equal bit for bit.)
template <class T> __device__ __forceinline__ V3<T> strided_apply(const Rot<T>& R, V3<T> d, int u) {
    return u % STRIDED_BATCH == 0 ? step_apply<true>(R, d) : step_apply<false>(R, d);
}

// F = sum f_j and tau = sum delta_j x f_j in FP64, delta_j = A(q)^T d_j
// Where body k (first atom atom0, N atoms) reads its body-fixed coordinates
// and inertia: its own, or, in a tile of bodies that share them, those of
// body DevSys::dOff[k] of the same size class, whose rows lie (k - ks) N rows
// before its own.  ks: the body whose 1/I and 1/M it reads; row: its first
// row of d.
struct Shape { int ks, row; };
__device__ __forceinline__ Shape body_shape(const DevSys& S, const Tile& tile, int k, int atom0, int N) {
    const int own = atom0 - S.numFree;
    if (!tile.sharedD) return {k, own};
    const int ks = S.dOff[k];
    return {ks, own - (k - ks) * N};
}

template <class Real, int NC, class IO>
__device__ __forceinline__ void body_sums(const DevSys& S, const Rot<Real>& R, int atom0, int dbase, int N, int sub,
                                          int lanes, V3<double>& F, V3<double>& tau) {
    if constexpr (NC > 0) {
        V3<Real> dj[NC], fj[NC];
#pragma unroll
        for (int j = 0; j < NC; j++) {
            dj[j] = ld3<Real>(S.d, S.dStride, dbase + j);
            fj[j] = IO::template force<Real>(S, atom0 + j);
        }
#pragma unroll
        for (int j = 0; j < NC; j++) {
            V3<double> dl = cvt<double>(step_apply<true>(R, dj[j]));
            V3<double> f = cvt<double>(fj[j]);
            F = F + f;
            tau = tau + cross(dl, f);
        }
    } else {
        // atoms sub, sub + lanes, ...: up to STRIDED_BATCH per lane loaded
        // before any is summed (one round trip for the bodies the default
        // lanes give), summed in the same order
        constexpr int U = STRIDED_BATCH;
        for (int j0 = sub; j0 < N; j0 += U * lanes) {
            V3<Real> dj[U], fj[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int j = j0 + u * lanes;
                if (j < N) {
                    dj[u] = ld3<Real>(S.d, S.dStride, dbase + j);
                    fj[u] = IO::template force<Real>(S, atom0 + j);
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (j0 + u * lanes < N) {
                    V3<double> dl = cvt<double>(strided_apply(R, dj[u], u));
                    V3<double> f = cvt<double>(fj[u]);
                    F = F + f;
                    tau = tau + cross(dl, f);
                }
            }
        }
    }
}

template <class Real, class IO = SoaAtoms>
__device__ __forceinline__ void body_sums_any(const DevSys& S, const Rot<Real>& R, int atom0, int dbase, int N,
                                              int sub, int lanes, bool active, V3<double>& F, V3<double>& tau) {
    F = {0.0, 0.0, 0.0};
    tau = {0.0, 0.0, 0.0};
    if (lanes == 1) {
        if (active) {
            switch (N) {
            case 2: body_sums<Real, 2, IO>(S, R, atom0, dbase, N, 0, 1, F, tau); break;
            case 3: body_sums<Real, 3, IO>(S, R, atom0, dbase, N, 0, 1, F, tau); break;
            case 4: body_sums<Real, 4, IO>(S, R, atom0, dbase, N, 0, 1, F, tau); break;
            case 6: body_sums<Real, 6, IO>(S, R, atom0, dbase, N, 0, 1, F, tau); break;
            default: body_sums<Real, 0, IO>(S, R, atom0, dbase, N, 0, 1, F, tau); break;
            }
        }
    } else {
        if (active) body_sums<Real, 0, IO>(S, R, atom0, dbase, N, sub, lanes, F, tau);
        F = {xor_sum(F.x, lanes), xor_sum(F.y, lanes), xor_sum(F.z, lanes)};
        tau = {xor_sum(tau.x, lanes), xor_sum(tau.y, lanes), xor_sum(tau.z, lanes)};
    }
}

// atom positions r_cm + A(q)^T d_j: fp32 in mixed precision (the force field's
// view; the exact value is rebuilt from the body state on download).  Bodies
// of 2 and 3 atoms, which lie in a plane of their principal axes, are placed
// with the y products rounded, as part 1 always placed them in adopted arrays,
// which show the last bit of the offset.
template <class Real, bool EXACT, int NC, class IO>
__device__ __forceinline__ void body_positions(const DevSys& S, const Rot<Real>& R, V3<double> rc, int atom0,
                                               int dbase, int N, int sub, int lanes) {
    if constexpr (NC > 0) {
        V3<Real> dj[NC];
        int at[NC];
#pragma unroll
        for (int j = 0; j < NC; j++) {
            dj[j] = ld3<Real>(S.d, S.dStride, dbase + j);
            at[j] = IO::at(S, atom0 + j);
        }
#pragma unroll
        for (int j = 0; j < NC; j++)
            IO::template set_body_pos_at<Real>(S, at[j],
                                               rc + cvt<double>(place_apply<(!EXACT && NC == 4)>(R, dj[j])));
    } else {
        // loads of a batch first, then its stores (one round trip per batch)
        constexpr int U = STRIDED_BATCH;
        for (int j0 = sub; j0 < N; j0 += U * lanes) {
            V3<Real> dj[U];
            int at[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                if (j0 + u * lanes < N) {
                    dj[u] = ld3<Real>(S.d, S.dStride, dbase + j0 + u * lanes);
                    at[u] = IO::at(S, atom0 + j0 + u * lanes);
                }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (j0 + u * lanes < N)
                    IO::template set_body_pos_at<Real>(S, at[u], rc + cvt<double>(strided_apply(R, dj[u], u)));
        }
    }
}

template <class Real, bool EXACT, class IO>
__device__ __forceinline__ void body_positions_any(const DevSys& S, const Rot<Real>& R, V3<double> rc, int atom0,
                                                   int dbase, int N, int sub, int lanes) {
    if (lanes == 1) {
        switch (N) {
        case 2: body_positions<Real, EXACT, 2, IO>(S, R, rc, atom0, dbase, N, 0, 1); break;
        case 3: body_positions<Real, EXACT, 3, IO>(S, R, rc, atom0, dbase, N, 0, 1); break;
        case 4: body_positions<Real, EXACT, 4, IO>(S, R, rc, atom0, dbase, N, 0, 1); break;
        case 6: body_positions<Real, EXACT, 6, IO>(S, R, rc, atom0, dbase, N, 0, 1); break;
        default: body_positions<Real, EXACT, 0, IO>(S, R, rc, atom0, dbase, N, 0, 1); break;
        }
    } else {
        body_positions<Real, EXACT, 0, IO>(S, R, rc, atom0, dbase, N, sub, lanes);
    }
}

// v_cm + w x delta with its fused operations written out
template <class Real> __device__ __forceinline__ V3<Real> atom_velocity(V3<Real> vcm, V3<Real> ws, V3<Real> dl) {
    return {vcm.x + fma(ws.y, dl.z, -(ws.z * dl.y)), vcm.y + fma(ws.z, dl.x, -(ws.x * dl.z)),
            vcm.z + fma(ws.x, dl.y, -(ws.y * dl.x))};
}

// (d and the atoms' places read before the first store, which they may alias:
// part 2 at 1M waters 29.0 -> 26.3 us)
template <class Real, int NC, class IO>
__device__ __forceinline__ void body_velocities(const DevSys& S, const Rot<Real>& R, V3<Real> vcm, V3<Real> ws,
                                                int atom0, int dbase, int N, int sub, int lanes) {
    if constexpr (NC > 0) {
        V3<Real> dj[NC];
        int at[NC];
#pragma unroll
        for (int j = 0; j < NC; j++) {
            dj[j] = ld3<Real>(S.d, S.dStride, dbase + j);
            at[j] = IO::at(S, atom0 + j);
        }
#pragma unroll
        for (int j = 0; j < NC; j++)
            IO::template set_vel_at<Real>(S, at[j], atom_velocity(vcm, ws, step_apply<true>(R, dj[j])));
    } else {
        constexpr int U = STRIDED_BATCH;
        for (int j0 = sub; j0 < N; j0 += U * lanes) {
            V3<Real> dj[U];
            int at[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                if (j0 + u * lanes < N) {
                    dj[u] = ld3<Real>(S.d, S.dStride, dbase + j0 + u * lanes);
                    at[u] = IO::at(S, atom0 + j0 + u * lanes);
                }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (j0 + u * lanes < N)
                    IO::template set_vel_at<Real>(S, at[u], atom_velocity(vcm, ws, strided_apply(R, dj[u], u)));
        }
    }
}
// A(q) x from the rows of A(q)^T, fused operations written out as in
// step_apply: the y product rounded, or, in the fused pass, the x product for
// the bodies that its NO-SQUISH form keeps in registers (one lane, 2 to 4
// atoms; an FP64 unit in the last place of a torque's moment)
template <class Real> __device__ __forceinline__ V3<double> to_body(const Rot<Real>& R, V3<double> x, bool small) {
    const V3<double> r0 = cvt<double>(R.r0), r1 = cvt<double>(R.r1), r2 = cvt<double>(R.r2);
    if (small)
        return {fma(r2.x, x.z, fma(r1.x, x.y, r0.x * x.x)), fma(r2.y, x.z, fma(r1.y, x.y, r0.y * x.x)),
                fma(r2.z, x.z, fma(r1.z, x.y, r0.z * x.x))};
    return {fma(r2.x, x.z, fma(r0.x, x.x, r1.x * x.y)), fma(r2.y, x.z, fma(r0.y, x.x, r1.y * x.y)),
            fma(r2.z, x.z, fma(r0.z, x.x, r1.z * x.y))};
}
// p + F h, fused
__device__ __forceinline__ V3<double> kicked(V3<double> p, V3<double> F, double h) {
    return {fma(F.x, h, p.x), fma(F.y, h, p.y), fma(F.z, h, p.z)};
}
__device__ __forceinline__ bool small_body(const DevSys& S, int N, int lanes) {
    return S.rotationMode != 0 && lanes == 1 && N <= 4;
}

// body-frame torque; a linear body (1/I2 = 0) has no moment about its axis
// and keeps L2 = 0 exactly (the axial torque of collinear atoms is rounding)
template <class Real> __device__ __forceinline__ V3<double> axial_torque(V3<double> tb, V3<Real> invI) {
    if (invI.z == (Real)0) tb.z = 0.0;
    return tb;
}

// free rotation of (q, L) over h: the FP64 exact solution or NO-SQUISH(mode)
template <class Real, bool EXACT>
__device__ __forceinline__ void free_rotation(Q4<Real>& q, V3<Real>& L, V3<Real> invI, double h, int mode) {
    if (EXACT) {
        Q4<double> qd = cvt<double>(q);
        V3<double> Ld = cvt<double>(L), invId = cvt<double>(invI);
        if (invI.z == (Real)0) {
            linear_rotor_exact(qd, Ld, invId, h);
        } else {
            V3<double> I = {1.0 / invId.x, 1.0 / invId.y, 1.0 / invId.z};
            exact_rotation<sizeof(Real) == 4>(qd, Ld, I, invId, h);
        }
        q = cvt<Real>(qd);
        L = cvt<Real>(Ld);
    } else {
        no_squish<Real>(q, L, invI, h, mode);
    }
}

// r_cm += p_cm (dt / M), then the free rotation of (q, L)
template <class Real, bool EXACT>
__device__ __forceinline__ void drift_and_rotate(const DevSys& S, Body<Real>& B, V3<double>& rc) {
    double idt = (double)B.invM * S.dt;
    rc = rc + cvt<double>(B.p) * idt;
    free_rotation<Real, EXACT>(B.q, B.L, B.invI, S.dt, S.rotationMode);
}

template <class Real> __device__ __forceinline__ void store_rcm(const DevSys& S, int k, V3<double> rc) {
    const int st = S.bodyStride;
    S.rcm[k] = rc.x;
    S.rcm[k + st] = rc.y;
    S.rcm[k + 2 * st] = rc.z;
}
template <class Real> __device__ __forceinline__ V3<double> load_rcm(const DevSys& S, int k) {
    const int st = S.bodyStride;
    return V3<double>{S.rcm[k], S.rcm[k + st], S.rcm[k + 2 * st]};
}

// ---------------------------------------------------------------------------
// part 1
// ---------------------------------------------------------------------------
// free-atom tiles hold up to FREE_PER_THREAD atoms per thread (strided by
// the workgroup size, so each pass over the tile is coalesced): load(u, a) for
// U of a thread's atoms, then use(u, a) for them
template <int U, class Load, class Use>
__device__ __forceinline__ void over_tile(const Tile& tile, Load&& load, Use&& use) {
    const int step = blockDim.x;
    for (int i0 = threadIdx.x; i0 < tile.count; i0 += U * step) {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i0 + u * step < tile.count) load(u, tile.first + i0 + u * step);
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i0 + u * step < tile.count) use(u, tile.first + i0 + u * step);
    }
}
// a batch of free atoms as a step reads them
template <class Real, class IO, int U> struct FreeBatch {
    int at[U];
    V3<Real> v[U], f[U];
    Real invm[U];
    __device__ __forceinline__ void load(const DevSys& S, int u, int a) {
        at[u] = IO::at(S, a);
        v[u] = IO::template vel_at<Real>(S, at[u]);
        f[u] = IO::template force_at<Real>(S, at[u]);
        invm[u] = reinterpret_cast<const Real*>(S.freeInvM)[a];
    }
};

template <class Real, class IO>
__device__ __forceinline__ void part1_free(const DevSys& S, const Tile& tile) {
    const Real halfDt = (Real)(0.5 * S.dt);
    constexpr int U = free_batch<Real, IO>();
    FreeBatch<Real, IO, U> atoms;
    V3<double> r[U];
    over_tile<U>(tile, [&](int u, int a) {
        atoms.load(S, u, a);
        r[u] = IO::template pos_at<Real>(S, atoms.at[u]);
    }, [&](int u, int a) {
        V3<Real> v = atoms.v[u] + atoms.f[u] * atoms.invm[u] * halfDt;
        V3<double> x = r[u] + cvt<double>(v) * S.dt;
        if constexpr (IO::adopted) {
            if (S.posDelta) {
                // the caller's constrained displacement; the correction to
                // the unconstrained drift waits for part 2
                const double* pd = S.posDelta + 4 * (size_t)atoms.at[u];
                const V3<double> ru = x;
                x = r[u] + V3<double>{pd[0], pd[1], pd[2]};
                st3<Real>(S.freeCorr, S.numFree, a, cvt<Real>(x - ru));
            }
        }
        IO::template set_vel_at<Real>(S, atoms.at[u], v);
        IO::template set_pos_at<Real>(S, atoms.at[u], x);
    });
}

// The free atoms' drift displacements (v + F (1/m) dt/2) dt, as part 1
// computes them, into a caller's posDelta (double4 per slot, w = 0) for its
// constraint solver (the CUDA platform's freeAtomsDelta,
// rigidbodyintegrator.cu:270-279); adopted arrays only.
template <class Real>
__global__ void k_free_delta(const DevSys* __restrict__ sys, double* __restrict__ posDelta) {
    const DevSys& S = *sys;
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= S.numFree) return;
    const Real halfDt = (Real)(0.5 * S.dt);
    V3<Real> v = AdoptedAtoms::vel<Real>(S, a);
    V3<Real> f = AdoptedAtoms::force<Real>(S, a);
    const Real invm = reinterpret_cast<const Real*>(S.freeInvM)[a];
    v = v + f * invm * halfDt;
    const V3<double> d = cvt<double>(v) * S.dt;
    double* o = posDelta + 4 * (size_t)S.ommSlot[a];
    o[0] = d.x;
    o[1] = d.y;
    o[2] = d.z;
    o[3] = 0.0;
}

template <class Real, bool EXACT, class IO>
__device__ __forceinline__ void part1_bodies(const DevSys& S, const Tile& tile) {
    const int shift = lane_shift(tile.lanes);
    const int b = threadIdx.x >> shift;
    const int sub = threadIdx.x & (tile.lanes - 1);
    if (b >= tile.count) return;
    const int k = tile.first + b;
    const int atom0 = tile.atomFirst + b * tile.N;
    const Shape sh = body_shape(S, tile, k, atom0, tile.N);
    const int dbase = sh.row;
    Body<Real> B = load_body<Real>(S, k, sh.ks);
    V3<double> rc = load_rcm<Real>(S, k);
    drift_and_rotate<Real, EXACT>(S, B, rc);
    auto store = [&] {
        if (sub == 0) {
            st4<Real>(S.q, k, B.q);
            stp3<Real>(S.L, k, B.L);
            store_rcm<Real>(S, k, rc);
        }
    };
    // adopted arrays: the state last, since the loads of the atoms' places
    // would wait behind it; the library's own: first, which leaves the
    // positions' registers free (1M waters 31.9 us, 34.4 with the state last)
    if (!IO::adopted) store();
    body_positions_any<Real, EXACT, IO>(S, step_rot(B.q), rc, atom0, dbase, tile.N, sub, tile.lanes);
    if (IO::adopted) store();
}

// How a step kernel holds its system descriptor.  The exact-rotation kernels
// take a register copy: read through the descriptor table, its fields are
// re-read after stores that may alias the table, and each re-read waits for
// the loads in flight (heterogeneous 200k system: fused pass 22.1 -> 21.7
// us).  The NO-SQUISH kernels keep the reference: the copy's scalar
// registers spill into vector ones and cost the fused pass a wave per SIMD.
template <bool COPY> using SysView = std::conditional_t<COPY, const DevSys, const DevSys&>;

template <class Real, bool EXACT, class IO>
__global__ __launch_bounds__(EXACT ? 256 : 512) void k_part1(const DevSys* __restrict__ systems,
                                                              const Tile* __restrict__ tiles, int numTiles) {
    for (int t = blockIdx.x; t < numTiles; t += gridDim.x) {
        const Tile tile = tiles[t];
        SysView<EXACT> S = systems[tile.sys];
        if (tile.kind == TILE_FREE)
            part1_free<Real, IO>(S, tile);
        else
            part1_bodies<Real, EXACT, IO>(S, tile);
    }
}

// ---------------------------------------------------------------------------
// part 2
// ---------------------------------------------------------------------------
template <class Real, class IO>
__device__ __forceinline__ void part2_free(const DevSys& S, const Tile& tile, double (&ke)[2]) {
    const Real halfDt = (Real)(0.5 * S.dt);
    constexpr int U = free_batch<Real, IO>();
    FreeBatch<Real, IO, U> atoms;
    over_tile<U>(tile, [&](int u, int a) { atoms.load(S, u, a); }, [&](int u, int a) {
        V3<Real> v = atoms.v[u] + atoms.f[u] * atoms.invm[u] * halfDt;
        // (R - saved) / dt of a constrained part 1
        if (IO::adopted && S.corrPending) v = v + ld3<Real>(S.freeCorr, S.numFree, a) * (Real)(1.0 / S.dt);
        IO::template set_vel_at<Real>(S, atoms.at[u], v);
        V3<double> vd = cvt<double>(v);
        ke[0] += dot(vd, vd) / (double)atoms.invm[u];
    });
}

template <class Real, class IO>
__device__ __forceinline__ void part2_bodies(const DevSys& S, const Tile& tile, double (&ke)[2]) {
    const int shift = lane_shift(tile.lanes);
    const int b = threadIdx.x >> shift;
    const int sub = threadIdx.x & (tile.lanes - 1);
    const bool active = b < tile.count;
    const int k = tile.first + (active ? b : 0);
    const int N = tile.N;
    const int atom0 = tile.atomFirst + (active ? b : 0) * N;
    const Shape sh = body_shape(S, tile, k, atom0, N);
    const int dbase = sh.row;
    Body<Real> B = load_body<Real>(S, k, sh.ks);
    Rot<Real> R = step_rot(B.q);
    V3<double> F, tau;
    body_sums_any<Real, IO>(S, R, atom0, dbase, N, sub, tile.lanes, active, F, tau);
    if (!active) return;
    const double halfDt = 0.5 * S.dt;
    V3<double> tb = axial_torque(to_body(R, tau, false), B.invI);
    V3<double> p = kicked(cvt<double>(B.p), F, halfDt);
    V3<double> L = kicked(cvt<double>(B.L), tb, halfDt);
    V3<double> w = hadamard(cvt<double>(B.invI), L);
    V3<double> vcm = p * (double)B.invM;
    const V3<Real> ws = step_apply<true>(R, cvt<Real>(w)), vc = cvt<Real>(vcm);
    switch (tile.lanes == 1 ? N : 0) {
    case 2: body_velocities<Real, 2, IO>(S, R, vc, ws, atom0, dbase, N, 0, 1); break;
    case 3: body_velocities<Real, 3, IO>(S, R, vc, ws, atom0, dbase, N, 0, 1); break;
    case 4: body_velocities<Real, 4, IO>(S, R, vc, ws, atom0, dbase, N, 0, 1); break;
    case 6: body_velocities<Real, 6, IO>(S, R, vc, ws, atom0, dbase, N, 0, 1); break;
    default: body_velocities<Real, 0, IO>(S, R, vc, ws, atom0, dbase, N, sub, tile.lanes); break;
    }
    if (sub == 0) {
        ke[0] = dot(p, vcm);
        ke[1] = dot(L, w);
        // first half-kick of the next step (same F and torque), its product
        // rounded before it is added
        stp3<Real>(S.pcm, k, cvt<Real>(p + scaled(F, halfDt)));
        stp3<Real>(S.L, k, cvt<Real>(L + scaled(tb, halfDt)));
    }
}

template <class Real, class IO>
__global__ __launch_bounds__(512) void k_part2(const DevSys* __restrict__ systems, const Tile* __restrict__ tiles,
                                                int numTiles) {
    for (int t = blockIdx.x; t < numTiles; t += gridDim.x) {
        const Tile tile = tiles[t];
        const DevSys& S = systems[tile.sys];
        double ke[2] = {0.0, 0.0};
        if (tile.kind == TILE_FREE)
            part2_free<Real, IO>(S, tile, ke);
        else
            part2_bodies<Real, IO>(S, tile, ke);
        block_reduce_store<2>(ke, S.kePart, tile.slot);
    }
}

// ---------------------------------------------------------------------------
// fused step boundary: part2 of step n followed by part1 of step n+1 for the
// same body, one pass over its data.  Inside RigidBodyIntegrator::step(k) the
// atom velocities and kinetic energies of the interior steps are read by
// nothing (forces depend on positions only), so this pass writes neither;
// the last step of the call ends with a plain part2.  The body state is
// rounded to storage precision at the same points as part2 + part1.
// ---------------------------------------------------------------------------
template <class Real, class IO>
__device__ __forceinline__ void fused_free(const DevSys& S, const Tile& tile) {
    const Real halfDt = (Real)(0.5 * S.dt);
    constexpr int U = free_batch<Real, IO>();
    FreeBatch<Real, IO, U> atoms;
    V3<double> r[U];
    over_tile<U>(tile, [&](int u, int a) {
        atoms.load(S, u, a);
        r[u] = IO::template pos_at<Real>(S, atoms.at[u]);
    }, [&](int u, int) {
        V3<Real> v = atoms.v[u];
        v = v + atoms.f[u] * atoms.invm[u] * halfDt;     // end of step n
        v = v + atoms.f[u] * atoms.invm[u] * halfDt;     // start of step n+1
        IO::template set_vel_at<Real>(S, atoms.at[u], v);
        IO::template set_pos_at<Real>(S, atoms.at[u], r[u] + cvt<double>(v) * S.dt);
    });
}

// part2 of step n and the first half-kick of step n+1 on the body momenta
template <class Real>
__device__ __forceinline__ void fused_kicks(const DevSys& S, Body<Real>& B, const Rot<Real>& R, V3<double> F,
                                            V3<double> tau, bool small) {
    const double halfDt = 0.5 * S.dt;
    V3<double> tb = axial_torque(to_body(R, tau, small), B.invI);
    V3<double> p = kicked(cvt<double>(B.p), F, halfDt);
    V3<double> L = kicked(cvt<double>(B.L), tb, halfDt);
    B.p = cvt<Real>(kicked(p, F, halfDt));
    B.L = cvt<Real>(kicked(L, tb, halfDt));
}

template <class Real> __device__ __forceinline__ void store_body(const DevSys& S, int k, const Body<Real>& B,
                                                                 V3<double> rc) {
    st4<Real>(S.q, k, B.q);
    stp3<Real>(S.L, k, B.L);
    stp3<Real>(S.pcm, k, B.p);
    store_rcm<Real>(S, k, rc);
}

// one lane per body of NC atoms: the body-fixed coordinates stay in registers
// from the torque sum to the position rebuild, so d is read once
template <class Real, bool EXACT, int NC, class IO>
__device__ __forceinline__ void fused_body_regs(const DevSys& S, int k, int atom0, int ks, int dbase) {
    Body<Real> B = load_body<Real>(S, k, ks);
    V3<double> rc = load_rcm<Real>(S, k);
    V3<Real> dj[NC], fj[NC];
    int at[NC];
#pragma unroll
    for (int j = 0; j < NC; j++) {
        dj[j] = ld3<Real>(S.d, S.dStride, dbase + j);
        at[j] = IO::at(S, atom0 + j);
        fj[j] = IO::template force_at<Real>(S, at[j]);
    }
    Rot<Real> R = step_rot(B.q);
    V3<double> F = {0.0, 0.0, 0.0}, tau = {0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < NC; j++) {
        V3<double> dl = cvt<double>(step_apply<true>(R, dj[j]));
        V3<double> f = cvt<double>(fj[j]);
        F = F + f;
        tau = tau + cross(dl, f);
    }
    fused_kicks<Real>(S, B, R, F, tau, true);
    drift_and_rotate<Real, EXACT>(S, B, rc);
    store_body<Real>(S, k, B, rc);
    Rot<Real> R1 = step_rot(B.q);
#pragma unroll
    for (int j = 0; j < NC; j++)
        IO::template set_body_pos_at<Real>(S, at[j], rc + cvt<double>(place_apply<!EXACT>(R1, dj[j])));
}

template <class Real, bool EXACT, class IO>
__device__ __forceinline__ void fused_bodies(const DevSys& S, const Tile& tile) {
    const int N = tile.N;
    // (the FP64 exact rotation leaves no registers to spare: it re-reads d)
    if (!EXACT && tile.lanes == 1 && (N == 2 || N == 3 || N == 4)) {
        const int b = threadIdx.x;
        if (b >= tile.count) return;
        const int k = tile.first + b, atom0 = tile.atomFirst + b * N;
        const Shape sh = body_shape(S, tile, k, atom0, N);
        if (N == 2) fused_body_regs<Real, EXACT, 2, IO>(S, k, atom0, sh.ks, sh.row);
        else if (N == 3) fused_body_regs<Real, EXACT, 3, IO>(S, k, atom0, sh.ks, sh.row);
        else fused_body_regs<Real, EXACT, 4, IO>(S, k, atom0, sh.ks, sh.row);
        return;
    }
    const int shift = lane_shift(tile.lanes);
    const int b = threadIdx.x >> shift;
    const int sub = threadIdx.x & (tile.lanes - 1);
    const bool active = b < tile.count;
    const int k = tile.first + (active ? b : 0);
    const int atom0 = tile.atomFirst + (active ? b : 0) * N;
    const Shape sh = body_shape(S, tile, k, atom0, N);
    const int dbase = sh.row;
    Body<Real> B = load_body<Real>(S, k, sh.ks);
    V3<double> rc = load_rcm<Real>(S, k);
    Rot<Real> R = step_rot(B.q);
    V3<double> F, tau;
    body_sums_any<Real, IO>(S, R, atom0, dbase, N, sub, tile.lanes, active, F, tau);
    if (!active) return;
    fused_kicks<Real>(S, B, R, F, tau, small_body(S, N, tile.lanes));
    drift_and_rotate<Real, EXACT>(S, B, rc);
    body_positions_any<Real, EXACT, IO>(S, step_rot(B.q), rc, atom0, dbase, N, sub, tile.lanes);
    if (sub == 0) store_body<Real>(S, k, B, rc);
}

template <class Real, bool EXACT, class IO>
__global__ __launch_bounds__(EXACT ? 256 : 512) void k_fused(const DevSys* __restrict__ systems,
                                                              const Tile* __restrict__ tiles, int numTiles) {
    for (int t = blockIdx.x; t < numTiles; t += gridDim.x) {
        const Tile tile = tiles[t];
        SysView<EXACT> S = systems[tile.sys];
        if (tile.kind == TILE_FREE)
            fused_free<Real, IO>(S, tile);
        else
            fused_bodies<Real, EXACT, IO>(S, tile);
    }
}

// ---------------------------------------------------------------------------
// Refined energies: the CUDA platform's COMPMOD terms
// (platforms/cuda/src/kernels/rigidbodyintegrator.cu:270-292, 318-320,
// 380-383, 433-469).  The accumulators of a step depend on that step alone,
// so they are evaluated for the last step of a call only, by two kernels
// that bracket it; the step kernels themselves are the same for every
// system.  In displacement form, equal in exact arithmetic to the
// reference's 2.5 r(t) + ... and 0.5 q(t-dt) - 3 q(t) + ...:
//   rdot = dt/2 [5 v(t+dt/2) - v(t-dt/2) + 2 v(t+3dt/2)]
//   qdot = (q(t-dt) - q(t))/2 + 5 (q(t+dt) - q(t))/2 + (q(t+2dt) - q(t+dt))
// where q(t-dt) and q(t+2dt) are virtual rotations from (q, L -/+ the
// torque half-kick) over -/+dt.  Free atoms use posDot = 2 rdot of the same
// form (with the sign of v(t-dt/2) the body terms have).
//   k_refine_begin, before the step: from its starting state and the
//     current forces, a_r = 5 p(t+dt/2) - p(t-dt/2) and the two q(t) terms
//     a_q per body (q(t+dt) by the step's own kick and rotation), and
//     a_v = 5 v(t+dt/2) - v(t-dt/2) per free atom.  `folded` = the stored
//     momenta carry the step's first half-kick (after part2 or the set-up);
//     otherwise the step is a fused boundary, which applies both half-kicks.
//   k_refine_end, after the step's part2: per tile
//     [0] sum m dt/2 (a + 2 v(t+3dt/2)) . v(t+dt)   (= 6 dt KE_t refined)
//     [1] sum qdot . pi(t+dt), pi = 2 B(q) L         (= 6 dt KE_r refined)
//     (qdot's component along q, which the reference projects out, has no
//     effect: B(q)^T q = 0).
// ---------------------------------------------------------------------------
template <class Real> __device__ __forceinline__ void store_refine_body(const DevSys& S, int k, V3<double> ar,
                                                                        Q4<double> aq) {
    st4<Real>(S.refBody, 2 * k, Q4<Real>{(Real)ar.x, (Real)ar.y, (Real)ar.z, (Real)0});
    st4<Real>(S.refBody, 2 * k + 1, cvt<Real>(aq));
}

template <class Real, class IO>
__device__ __forceinline__ void refine_begin_free(const DevSys& S, const Tile& tile, bool folded) {
    Real halfDt = (Real)(0.5 * S.dt);
    for (int i = threadIdx.x; i < tile.count; i += blockDim.x) {
        int a = tile.first + i;
        V3<Real> v = IO::template vel<Real>(S, a);
        V3<Real> f = IO::template force<Real>(S, a);
        Real invm = reinterpret_cast<const Real*>(S.freeInvM)[a];
        V3<Real> dv = f * invm * halfDt;
        V3<double> av;
        if (folded) {   // v = v(t): 5 (v + dv) - (v - dv)
            av = cvt<double>(v) * 4.0 + cvt<double>(dv) * 6.0;
        } else {        // v = v(t-dt/2), v(t+dt/2) as the fused boundary forms it
            V3<Real> vp = v + dv;
            vp = vp + dv;
            av = cvt<double>(vp) * 5.0 + cvt<double>(v) * -1.0;
        }
        stp3<Real>(S.refFree, a, cvt<Real>(av));
    }
}

template <class Real, bool EXACT, class IO>
__device__ __forceinline__ void refine_begin_bodies(const DevSys& S, const Tile& tile, bool folded) {
    const int shift = lane_shift(tile.lanes);
    const int b = threadIdx.x >> shift;
    const int sub = threadIdx.x & (tile.lanes - 1);
    const bool active = b < tile.count;
    const int k = tile.first + (active ? b : 0);
    const int atom0 = tile.atomFirst + (active ? b : 0) * tile.N;
    const Shape sh = body_shape(S, tile, k, atom0, tile.N);
    Body<Real> B = load_body<Real>(S, k, sh.ks);
    Rot<Real> R = step_rot(B.q);
    V3<double> F, tau;
    body_sums_any<Real, IO>(S, R, atom0, sh.row, tile.N, sub, tile.lanes, active, F, tau);
    if (!active || sub != 0) return;
    V3<double> tb = axial_torque(to_body(R, tau, false), B.invI);
    V3<double> ar;
    V3<Real> Lback;
    Body<Real> B1 = B;
    if (folded) {
        // stored p = p(t+dt/2), L = L(t) + tau dt/2
        ar = cvt<double>(B.p) * 4.0 + F * S.dt;
        Lback = cvt<Real>(cvt<double>(B.L) + tb * -S.dt);
    } else {
        // stored p = p(t-dt/2), L = L(t) - tau dt/2 (after the last rotation)
        fused_kicks<Real>(S, B1, R, F, tau, false);
        ar = cvt<double>(B1.p) * 5.0 + cvt<double>(B.p) * -1.0;
        Lback = B.L;
    }
    Q4<Real> qm = B.q;
    free_rotation<Real, EXACT>(qm, Lback, B.invI, -S.dt, S.rotationMode);
    free_rotation<Real, EXACT>(B1.q, B1.L, B.invI, S.dt, S.rotationMode);
    Q4<double> q0 = cvt<double>(B.q) * -1.0;
    Q4<double> aq = (cvt<double>(qm) + q0) * 0.5 + (cvt<double>(B1.q) + q0) * 2.5;
    store_refine_body<Real>(S, k, ar, aq);
}

template <class Real, bool EXACT, class IO>
__global__ __launch_bounds__(EXACT ? 256 : 512) void k_refine_begin(const DevSys* __restrict__ systems,
                                                                     const Tile* __restrict__ tiles, int numTiles,
                                                                     int folded) {
    for (int t = blockIdx.x; t < numTiles; t += gridDim.x) {
        const Tile tile = tiles[t];
        const DevSys& S = systems[tile.sys];
        if (!S.refBody) continue;
        if (tile.kind == TILE_FREE)
            refine_begin_free<Real, IO>(S, tile, folded != 0);
        else
            refine_begin_bodies<Real, EXACT, IO>(S, tile, folded != 0);
    }
}

template <class Real, class IO>
__device__ __forceinline__ void refine_end_free(const DevSys& S, const Tile& tile, double (&rk)[2]) {
    const double halfDt = 0.5 * S.dt;
    for (int i = threadIdx.x; i < tile.count; i += blockDim.x) {
        int a = tile.first + i;
        V3<double> v = cvt<double>(IO::template vel<Real>(S, a));
        V3<double> f = cvt<double>(IO::template force<Real>(S, a));
        double invm = (double)reinterpret_cast<const Real*>(S.freeInvM)[a];
        // posDot / dt = a_v + 2 v(t+3dt/2)
        V3<double> pd = cvt<double>(ldp3<Real>(S.refFree, a)) + (v + f * (invm * halfDt)) * 2.0;
        rk[0] += 0.5 * S.dt * dot(pd, v) / invm;
    }
}

template <class Real, bool EXACT, class IO>
__device__ __forceinline__ void refine_end_bodies(const DevSys& S, const Tile& tile, double (&rk)[2]) {
    const int shift = lane_shift(tile.lanes);
    const int b = threadIdx.x >> shift;
    const int sub = threadIdx.x & (tile.lanes - 1);
    const bool active = b < tile.count;
    const int k = tile.first + (active ? b : 0);
    const int atom0 = tile.atomFirst + (active ? b : 0) * tile.N;
    // stored after part2: q(t+dt), p and L with the next half-kick folded in
    const Shape sh = body_shape(S, tile, k, atom0, tile.N);
    Body<Real> B = load_body<Real>(S, k, sh.ks);
    Rot<Real> R = step_rot(B.q);
    V3<double> F, tau;
    body_sums_any<Real, IO>(S, R, atom0, sh.row, tile.N, sub, tile.lanes, active, F, tau);
    if (!active || sub != 0) return;
    const double halfDt = 0.5 * S.dt;
    V3<double> tb = axial_torque(to_body(R, tau, false), B.invI);
    V3<double> p1 = cvt<double>(B.p) + F * -halfDt;
    V3<double> L1 = cvt<double>(B.L) + tb * -halfDt;
    Q4<Real> r0 = ld4<Real>(S.refBody, 2 * k), r1 = ld4<Real>(S.refBody, 2 * k + 1);
    // M rdot . v = dt/2 (a_r + 2 p(t+3dt/2)) . p(t+dt) / M
    V3<double> ar = {(double)r0.a, (double)r0.b, (double)r0.c};
    rk[0] = 0.5 * S.dt * (double)B.invM * dot(ar + cvt<double>(B.p) * 2.0, p1);
    // q(t+2dt): the next step's rotation from (q, L + tau dt/2)
    Q4<Real> q2 = B.q;
    V3<Real> L2 = B.L;
    free_rotation<Real, EXACT>(q2, L2, B.invI, S.dt, S.rotationMode);
    Q4<double> q1 = cvt<double>(B.q);
    Q4<double> qdot = cvt<double>(r1) + cvt<double>(q2) + q1 * -1.0;
    rk[1] = 2.0 * dot(Btmul(q1, qdot), L1);
}

template <class Real, bool EXACT, class IO>
__global__ __launch_bounds__(EXACT ? 256 : 512) void k_refine_end(const DevSys* __restrict__ systems,
                                                                   const Tile* __restrict__ tiles, int numTiles) {
    for (int t = blockIdx.x; t < numTiles; t += gridDim.x) {
        const Tile tile = tiles[t];
        const DevSys& S = systems[tile.sys];
        if (!S.refBody) continue;
        double rk[2] = {0.0, 0.0};
        if (tile.kind == TILE_FREE)
            refine_end_free<Real, IO>(S, tile, rk);
        else
            refine_end_bodies<Real, EXACT, IO>(S, tile, rk);
        block_reduce_store<2>(rk, S.refKePart, tile.slot);
    }
}

// potential-energy refinement partials (rigidbodyintegrator.cu:449-469):
// sum |F|^2/m over free atoms and |F|^2/M + tau.(I^-1 tau) over bodies, with
// the body-frame torque tau = B(q)^T C(q) tau_space of the current forces
template <class Real, class IO>
__global__ __launch_bounds__(512) void k_refine_pe(const DevSys* __restrict__ systems,
                                                    const Tile* __restrict__ tiles, int numTiles) {
    for (int t = blockIdx.x; t < numTiles; t += gridDim.x) {
        const Tile tile = tiles[t];
        const DevSys& S = systems[tile.sys];
        if (!S.refPePart) continue;
        double u[1] = {0.0};
        if (tile.kind == TILE_FREE) {
            for (int i = threadIdx.x; i < tile.count; i += blockDim.x) {
                int a = tile.first + i;
                V3<double> f = cvt<double>(IO::template force<Real>(S, a));
                u[0] += dot(f, f) * (double)reinterpret_cast<const Real*>(S.freeInvM)[a];
            }
        } else {
            const int shift = lane_shift(tile.lanes);
            const int b = threadIdx.x >> shift;
            const int sub = threadIdx.x & (tile.lanes - 1);
            const bool active = b < tile.count;
            const int k = tile.first + (active ? b : 0);
            const int atom0 = tile.atomFirst + (active ? b : 0) * tile.N;
            const Shape sh = body_shape(S, tile, k, atom0, tile.N);
            Body<Real> B = load_body<Real>(S, k, sh.ks);
            Rot<Real> R = step_rot(B.q);
            V3<double> F, tau;
            body_sums_any<Real, IO>(S, R, atom0, sh.row, tile.N, sub, tile.lanes, active, F, tau);
            if (active && sub == 0) {
                V3<double> tb = axial_torque(to_body(R, tau, false), B.invI);
                u[0] = dot(F, F) * (double)B.invM + dot(hadamard(tb, cvt<double>(B.invI)), tb);
            }
        }
        block_reduce_store<1>(u, S.refPePart, tile.slot);
    }
}

// ---------------------------------------------------------------------------
// Distance constraints between free atoms.  The reference applies OpenMM's
// constraints to the positions after part 1 (the positions before the step
// give the bond directions) and to the velocities after part 2
// (ReferenceRigidBodyKernels.cpp:92-104); part 2's (r - saved)/dt term
// (RigidBodySystem.cpp:193-204) carries the position correction into the
// velocities.  One lane per cluster of constrained atoms: SHAKE (Ryckaert,
// Ciccotti and Berendsen 1977) and RATTLE's velocity stage (Andersen 1983),
// Gauss-Seidel over the cluster's constraints in the order given, in FP64.
// Positions are converged when every |r_ij| is within (1 +- tol) d_ij,
// velocities when every |r_ij . v_ij| <= tol |r_ij| |v_ij|.  The kicks and
// the kinetic energy are those of the unconstrained free atoms; the
// correction (r - r_drift)/dt is added right after SHAKE rather than in
// part 2 (nothing reads the velocities in between).
// ---------------------------------------------------------------------------
// Per-atom values of one cluster.  Clusters of NA <= 4 atoms (every tile
// holds clusters of one size) keep them in registers and reach atom i of a
// constraint by selects; larger ones index private memory.
template <int NA> struct ClusterSlots {
    V3<double> v[NA];
    __device__ __forceinline__ V3<double> get(int i) const {
        if constexpr (NA <= 4) {
            V3<double> o = v[0];
#pragma unroll
            for (int k = 1; k < NA; k++)
                if (i == k) o = v[k];
            return o;
        } else {
            return v[i];
        }
    }
    __device__ __forceinline__ void add(int i, V3<double> d) {
        if constexpr (NA <= 4) {
#pragma unroll
            for (int k = 0; k < NA; k++)
                if (i == k) v[k] = v[k] + d;
        } else {
            v[i] = v[i] + d;
        }
    }
};

// The constraints of one cluster: for NA <= 4 at most NA (NA - 1) / 2 (the
// distinct pairs), held in registers and read once per step; larger
// clusters read them from memory in every sweep.
template <int NA> struct ClusterCons {
    static constexpr int kMax = NA <= 4 ? NA * (NA - 1) / 2 : 1;
    // sweeps over the constraints unroll fully for the register classes; the
    // general class loops over its count
    static constexpr int kUnroll = NA <= 4 ? kMax : 1;
    int n = 0, k0 = 0, a0 = 0;
    int ci[kMax], cj[kMax];
    double cd[kMax];
    const DevSys* S = nullptr;
    __device__ __forceinline__ void load(const DevSys& sys, int first, int last, int atom0) {
        S = &sys;
        n = last - first;
        k0 = first;
        a0 = atom0;
        if constexpr (NA <= 4) {
#pragma unroll
            for (int k = 0; k < kMax; k++)
                if (k < n) {
                    ci[k] = sys.consA[first + k] - atom0;
                    cj[k] = sys.consB[first + k] - atom0;
                    cd[k] = sys.consDist[first + k];
                }
        }
    }
    // atoms and length of constraint k (0 <= k < n)
    __device__ __forceinline__ void get(int k, int& i, int& j, double& d) const {
        if constexpr (NA <= 4) {
            i = ci[k];
            j = cj[k];
            d = cd[k];
        } else {
            i = S->consA[k0 + k] - a0;
            j = S->consB[k0 + k] - a0;
            d = S->consDist[k0 + k];
        }
    }
};

template <int NA>
__device__ __forceinline__ bool shake(const DevSys& S, const ClusterCons<NA>& C, ClusterSlots<NA>& r, const ClusterSlots<NA>& ro,
                      const ClusterSlots<NA>& w) {
    const double lo = (1.0 - S.constraintTol) * (1.0 - S.constraintTol);
    const double hi = (1.0 + S.constraintTol) * (1.0 + S.constraintTol);
    for (int it = 0; it < CLUSTER_MAX_ITERATIONS; it++) {
        bool done = true;
#pragma unroll ClusterCons<NA>::kUnroll
        for (int k = 0; k < ClusterCons<NA>::kMax || NA > 4; k++) {
            if (k >= C.n) break;
            int i, j;
            double dist;
            C.get(k, i, j, dist);
            const double d2 = dist * dist;
            V3<double> s = r.get(i) - r.get(j);
            double s2 = dot(s, s);
            if (s2 >= lo * d2 && s2 <= hi * d2) continue;
            done = false;
            const double wi = w.get(i).x, wj = w.get(j).x;
            V3<double> b = ro.get(i) - ro.get(j);
            double g = (d2 - s2) / (2.0 * (wi + wj) * dot(s, b));
            r.add(i, b * (g * wi));
            r.add(j, b * (-(g * wj)));
        }
        if (done) return true;
    }
    return false;
}

template <int NA>
__device__ __forceinline__ bool rattle(const DevSys& S, const ClusterCons<NA>& C, const ClusterSlots<NA>& r, ClusterSlots<NA>& v,
                       const ClusterSlots<NA>& w) {
    const double tol2 = S.constraintTol * S.constraintTol;
    for (int it = 0; it < CLUSTER_MAX_ITERATIONS; it++) {
        bool done = true;
#pragma unroll ClusterCons<NA>::kUnroll
        for (int k = 0; k < ClusterCons<NA>::kMax || NA > 4; k++) {
            if (k >= C.n) break;
            int i, j;
            double dist;
            C.get(k, i, j, dist);
            V3<double> s = r.get(i) - r.get(j);
            V3<double> dv = v.get(i) - v.get(j);
            double rv = dot(s, dv), s2 = dot(s, s);
            if (rv * rv <= tol2 * s2 * dot(dv, dv)) continue;
            done = false;
            const double wi = w.get(i).x, wj = w.get(j).x;
            double g = -rv / ((wi + wj) * s2);
            v.add(i, s * (g * wi));
            v.add(j, s * (-(g * wj)));
        }
        if (done) return true;
    }
    return false;
}

// one cluster of n atoms (n == NA when NA <= 4, n <= NA otherwise)
template <class Real, int NA>
__device__ __forceinline__ void cluster_phase(const DevSys& S, int c, int phase, double (&ke)[2]) {
    const int a0 = S.clusterStart[c];
    const int n = NA <= 4 ? NA : S.clusterStart[c + 1] - a0;
    const Real* invm = reinterpret_cast<const Real*>(S.freeInvM);
    if (phase == CLUSTER_KE) {
        // after the set-up: as k_setup's free atoms (staged FP64 velocities)
        for (int j = 0; j < n; j++) {
            const int a = a0 + j;
            V3<double> v = S.useStageV ? V3<double>{S.stageV[3 * (size_t)a], S.stageV[3 * (size_t)a + 1],
                                                    S.stageV[3 * (size_t)a + 2]}
                                       : cvt<double>(ld3<Real>(S.vel, S.atomStride, a));
            ke[0] += dot(v, v) / (double)invm[a];
        }
        return;
    }
    const double dt = S.dt;
    const Real halfDt = (Real)(0.5 * dt);
    V3<Real> v[NA];
    ClusterSlots<NA> r, vd, w;   // w holds 1/m in x
    ClusterCons<NA> C;
    C.load(S, S.consStart[c], S.consStart[c + 1], a0);
#pragma unroll
    for (int j = 0; j < NA; j++) {
        if (NA > 4 && j >= n) break;
        v[j] = ld3<Real>(S.vel, S.atomStride, a0 + j);
        r.v[j] = load_pos<Real>(S, a0 + j);
        w.v[j] = V3<double>{1.0 / S.mass[a0 + j], 0.0, 0.0};
    }
    bool ok = true;
    if (phase == CLUSTER_PART2 || phase == CLUSTER_FUSED) {
#pragma unroll
        for (int j = 0; j < NA; j++) {
            if (NA > 4 && j >= n) break;
            V3<Real> f = ld3<Real>(S.force, S.atomStride, a0 + j);
            vd.v[j] = cvt<double>(v[j] + f * invm[a0 + j] * halfDt);
        }
        ok = rattle<NA>(S, C, r, vd, w) && ok;
#pragma unroll
        for (int j = 0; j < NA; j++) {
            if (NA > 4 && j >= n) break;
            v[j] = cvt<Real>(vd.v[j]);
            if (phase == CLUSTER_PART2) {
                V3<double> u = cvt<double>(v[j]);
                ke[0] += dot(u, u) / (double)invm[a0 + j];
            }
        }
    }
    if (phase == CLUSTER_PART1 || phase == CLUSTER_FUSED) {
        ClusterSlots<NA> ro, ru;   // before the step, after the drift
#pragma unroll
        for (int j = 0; j < NA; j++) {
            if (NA > 4 && j >= n) break;
            V3<Real> f = ld3<Real>(S.force, S.atomStride, a0 + j);
            v[j] = v[j] + f * invm[a0 + j] * halfDt;
            ro.v[j] = r.v[j];
            r.v[j] = r.v[j] + cvt<double>(v[j]) * dt;
            ru.v[j] = r.v[j];
        }
        ok = shake<NA>(S, C, r, ro, w) && ok;
        const double invDt = 1.0 / dt;
#pragma unroll
        for (int j = 0; j < NA; j++) {
            if (NA > 4 && j >= n) break;
            v[j] = cvt<Real>(cvt<double>(v[j]) + (r.v[j] - ru.v[j]) * invDt);
            store_pos<Real>(S, a0 + j, r.v[j]);
        }
    }
#pragma unroll
    for (int j = 0; j < NA; j++) {
        if (NA > 4 && j >= n) break;
        st3<Real>(S.vel, S.atomStride, a0 + j, v[j]);
    }
    if (!ok) atomicAdd(S.constraintFail, 1u);
}

// ---- clusters of NA = 2..4 atoms: every per-atom and per-constraint value
// is a named register reached by a compile-time index (an array indexed by
// the atom numbers of a constraint would go to private memory)
template <int... I, class F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

template <class T> struct Four {
    T e0, e1, e2, e3;
    template <int J> __device__ __forceinline__ T& at() {
        if constexpr (J == 0) return e0;
        else if constexpr (J == 1) return e1;
        else if constexpr (J == 2) return e2;
        else return e3;
    }
    // element i (0 <= i < NA) as a sum of the elements weighted by exact 0/1
    // factors (selects would be turned back into an indexed load)
    template <int NA> __device__ __forceinline__ T get(int i) const {
        T o = e0 * (double)(i == 0);
        if (NA > 1) o = o + e1 * (double)(i == 1);
        if (NA > 2) o = o + e2 * (double)(i == 2);
        if (NA > 3) o = o + e3 * (double)(i == 3);
        return o;
    }
    template <int NA> __device__ __forceinline__ void add(int i, T d) {
        e0 = e0 + d * (double)(i == 0);
        if (NA > 1) e1 = e1 + d * (double)(i == 1);
        if (NA > 2) e2 = e2 + d * (double)(i == 2);
        if (NA > 3) e3 = e3 + d * (double)(i == 3);
    }
};

// The constraints of a small cluster, at most NA (NA - 1) / 2.  With 2 and 3
// atoms the cluster's atoms are taken in an order in which constraint 0 joins
// A and B, 1 B and C, 2 A and C (whatever their order and sense in memory: a
// constraint's correction is the same bit for bit taken from either end), so
// that a sweep reaches every value at a compile-time index; with 4 atoms the
// atoms of a constraint are found by their numbers.  What bounds a sweep is
// the chain of FP64 operations from one constraint to the next: with every
// access by number, 54 operations of a correction's 110 only found its atoms
// (2000 triangles, a fused pass: 13.3 us by number, 10.5 in order).
template <int NA> struct SmallCons {
    static constexpr int kMax = NA * (NA - 1) / 2;
    static constexpr bool kOrdered = NA <= 3;
    int n;
    int ci[6], cj[6];   // (kOrdered: not kept)
    double cd[6];
};
// the atoms of constraint k
constexpr int kFirst[3] = {0, 1, 0}, kSecond[3] = {1, 2, 2};

template <int NA, int K, class T> __device__ __forceinline__ T first_of(const SmallCons<NA>& C, Four<T>& x) {
    if constexpr (SmallCons<NA>::kOrdered) return x.template at<kFirst[K]>();
    else return x.template get<NA>(C.ci[K]);
}
template <int NA, int K, class T> __device__ __forceinline__ T second_of(const SmallCons<NA>& C, Four<T>& x) {
    if constexpr (SmallCons<NA>::kOrdered) return x.template at<kSecond[K]>();
    else return x.template get<NA>(C.cj[K]);
}
// x_i += a, x_j += b for the atoms i and j of constraint K
template <int NA, int K>
__device__ __forceinline__ void correct(const SmallCons<NA>& C, Four<V3<double>>& x, V3<double> a, V3<double> b) {
    if constexpr (SmallCons<NA>::kOrdered) {
        x.template at<kFirst[K]>() = x.template at<kFirst[K]>() + a;
        x.template at<kSecond[K]>() = x.template at<kSecond[K]>() + b;
    } else {
        x.template add<NA>(C.ci[K], a);
        x.template add<NA>(C.cj[K], b);
    }
}

template <int NA>
__device__ __forceinline__ bool shake_small(const DevSys& S, const SmallCons<NA>& C, Four<V3<double>>& r,
                                            Four<V3<double>>& ro, Four<double>& w) {
    const double lo = (1.0 - S.constraintTol) * (1.0 - S.constraintTol);
    const double hi = (1.0 + S.constraintTol) * (1.0 + S.constraintTol);
    for (int it = 0; it < CLUSTER_MAX_ITERATIONS; it++) {
        bool done = true;
        static_for<SmallCons<NA>::kMax>([&](auto K) {
            constexpr int k = K;
            if (k >= C.n) return;
            const double d2 = product(C.cd[k], C.cd[k]);
            V3<double> s = first_of<NA, k>(C, r) - second_of<NA, k>(C, r);
            double s2 = step_dot<true>(s, s);
            if (s2 >= lo * d2 && s2 <= hi * d2) return;
            done = false;
            const double wi = first_of<NA, k>(C, w), wj = second_of<NA, k>(C, w);
            V3<double> b = first_of<NA, k>(C, ro) - second_of<NA, k>(C, ro);
            double g = (d2 - s2) / (2.0 * (wi + wj) * step_dot<true>(s, b));
            correct<NA, k>(C, r, scaled(b, g * wi), scaled(b, -(g * wj)));
        });
        if (done) return true;
    }
    return false;
}

template <int NA>
__device__ __forceinline__ bool rattle_small(const DevSys& S, const SmallCons<NA>& C, Four<V3<double>>& r,
                                             Four<V3<double>>& v, Four<double>& w) {
    const double tol2 = S.constraintTol * S.constraintTol;
    for (int it = 0; it < CLUSTER_MAX_ITERATIONS; it++) {
        bool done = true;
        static_for<SmallCons<NA>::kMax>([&](auto K) {
            constexpr int k = K;
            if (k >= C.n) return;
            V3<double> s = first_of<NA, k>(C, r) - second_of<NA, k>(C, r);
            V3<double> dv = first_of<NA, k>(C, v) - second_of<NA, k>(C, v);
            double rv = step_dot<false>(s, dv), s2 = step_dot<true>(s, s);
            if (rv * rv <= tol2 * s2 * step_dot<false>(dv, dv)) return;
            done = false;
            const double wi = first_of<NA, k>(C, w), wj = second_of<NA, k>(C, w);
            double g = -rv / ((wi + wj) * s2);
            correct<NA, k>(C, v, scaled(s, g * wi), scaled(s, -(g * wj)));
        });
        if (done) return true;
    }
    return false;
}

// v + a dt/2, fused
template <class Real> __device__ __forceinline__ V3<Real> half_kick(V3<Real> v, V3<Real> a, Real halfDt) {
    return {fma(a.x, halfDt, v.x), fma(a.y, halfDt, v.y), fma(a.z, halfDt, v.z)};
}
// a cluster of exactly NA atoms in registers
template <class Real, int NA> struct SmallCluster {
    Four<int> atom;
    SmallCons<NA> C;
    Four<V3<Real>> v;
    Four<V3<double>> r;
    Four<double> w;       // 1/m
    Four<Real> invm;

    __device__ __forceinline__ void load(const DevSys& S, int c) {
        const int a0 = S.clusterStart[c], k0 = S.consStart[c];
        C.n = S.consStart[c + 1] - k0;
        int ci[SmallCons<NA>::kMax], cj[SmallCons<NA>::kMax];
        static_for<SmallCons<NA>::kMax>([&](auto K) {
            constexpr int k = K;
            ci[k] = cj[k] = 0;
            if (k < C.n) {
                ci[k] = S.consA[k0 + k] - a0;
                cj[k] = S.consB[k0 + k] - a0;
                C.cd[k] = S.consDist[k0 + k];
                if constexpr (!SmallCons<NA>::kOrdered) {
                    C.ci[k] = ci[k];
                    C.cj[k] = cj[k];
                }
            }
        });
        if constexpr (NA == 3) {
            // C is not in constraint 0, B is C's partner in constraint 1
            const int c2 = 3 - ci[0] - cj[0], b = ci[1] + cj[1] - c2;
            atom = {a0 + 3 - b - c2, a0 + b, a0 + c2, 0};
        } else {
            atom = {a0, a0 + 1, a0 + 2, a0 + 3};
        }
        static_for<NA>([&](auto J) {
            constexpr int j = J;
            const int a = atom.template at<j>();
            v.template at<j>() = ld3<Real>(S.vel, S.atomStride, a);
            r.template at<j>() = load_pos<Real>(S, a);
            w.template at<j>() = 1.0 / S.mass[a];
            invm.template at<j>() = reinterpret_cast<const Real*>(S.freeInvM)[a];
        });
    }
    // the velocities' second half-kick and their constraints
    __device__ __forceinline__ bool end_step(const DevSys& S, Four<V3<Real>>& f) {
        const Real halfDt = (Real)(0.5 * S.dt);
        Four<V3<double>> vd;
        static_for<NA>([&](auto J) {
            constexpr int j = J;
            vd.template at<j>() = cvt<double>(half_kick(v.template at<j>(), f.template at<j>() * invm.template at<j>(), halfDt));
        });
        const bool ok = rattle_small<NA>(S, C, r, vd, w);
        static_for<NA>([&](auto J) { v.template at<(int)J>() = cvt<Real>(vd.template at<(int)J>()); });
        return ok;
    }
    // the first half-kick, the drift and the positions' constraints
    __device__ __forceinline__ bool begin_step(const DevSys& S, Four<V3<Real>>& f) {
        const Real halfDt = (Real)(0.5 * S.dt);
        Four<V3<double>> ro, ru;   // before the step, after the drift
        static_for<NA>([&](auto J) {
            constexpr int j = J;
            v.template at<j>() = half_kick(v.template at<j>(), f.template at<j>() * invm.template at<j>(), halfDt);
            ro.template at<j>() = r.template at<j>();
            r.template at<j>() = r.template at<j>() + cvt<double>(v.template at<j>()) * S.dt;
            ru.template at<j>() = r.template at<j>();
        });
        const bool ok = shake_small<NA>(S, C, r, ro, w);
        const double invDt = 1.0 / S.dt;
        static_for<NA>([&](auto J) {
            constexpr int j = J;
            v.template at<j>() =
                cvt<Real>(cvt<double>(v.template at<j>()) + (r.template at<j>() - ru.template at<j>()) * invDt);
        });
        return ok;
    }
    __device__ __forceinline__ Four<V3<Real>> stored_forces(const DevSys& S) {
        Four<V3<Real>> f;
        static_for<NA>([&](auto J) {
            f.template at<(int)J>() = ld3<Real>(S.force, S.atomStride, atom.template at<(int)J>());
        });
        return f;
    }
    __device__ __forceinline__ void store_positions(const DevSys& S) {
        static_for<NA>([&](auto J) { store_pos<Real>(S, atom.template at<(int)J>(), r.template at<(int)J>()); });
    }
    __device__ __forceinline__ void store_velocities(const DevSys& S) {
        static_for<NA>([&](auto J) {
            st3<Real>(S.vel, S.atomStride, atom.template at<(int)J>(), v.template at<(int)J>());
        });
    }
};

// the same steps as cluster_phase, for a cluster of exactly NA atoms
template <class Real, int NA>
__device__ __forceinline__ void cluster_phase_small(const DevSys& S, int c, int phase, double (&ke)[2]) {
    if (phase == CLUSTER_KE) {
        const int a0 = S.clusterStart[c];
        const Real* invm = reinterpret_cast<const Real*>(S.freeInvM);
        static_for<NA>([&](auto J) {
            const int a = a0 + (int)J;
            V3<double> v = S.useStageV ? V3<double>{S.stageV[3 * (size_t)a], S.stageV[3 * (size_t)a + 1],
                                                    S.stageV[3 * (size_t)a + 2]}
                                       : cvt<double>(ld3<Real>(S.vel, S.atomStride, a));
            ke[0] += dot(v, v) / (double)invm[a];
        });
        return;
    }
    SmallCluster<Real, NA> K;
    K.load(S, c);
    Four<V3<Real>> f = K.stored_forces(S);
    bool ok = true;
    if (phase == CLUSTER_PART2 || phase == CLUSTER_FUSED) ok = K.end_step(S, f) && ok;
    if (phase == CLUSTER_PART2) {
        static_for<NA>([&](auto J) {
            V3<double> u = cvt<double>(K.v.template at<(int)J>());
            ke[0] += dot(u, u) / (double)K.invm.template at<(int)J>();
        });
    } else {
        ok = K.begin_step(S, f) && ok;
        K.store_positions(S);
    }
    K.store_velocities(S);
    if (!ok) atomicAdd(S.constraintFail, 1u);
}

// tiles of clusters of NA = 2, 3 or 4 atoms (registers only), or of larger
// clusters (NA = CLUSTER_MAX_ATOMS, private memory)
template <class Real, int NA>
__global__ __launch_bounds__(256) void k_clusters(const DevSys* __restrict__ systems, const Tile* __restrict__ tiles,
                                                   int numTiles, int phase) {
    for (int t = blockIdx.x; t < numTiles; t += gridDim.x) {
        const Tile tile = tiles[t];
        const DevSys& S = systems[tile.sys];
        double ke[3] = {0.0, 0.0, 0.0};
        if ((int)threadIdx.x < tile.count) {
            double k2[2] = {0.0, 0.0};
            if constexpr (NA <= 4) cluster_phase_small<Real, NA>(S, tile.first + threadIdx.x, phase, k2);
            else cluster_phase<Real, NA>(S, tile.first + threadIdx.x, phase, k2);
            ke[0] = k2[0];
        }
        // set-up partials carry a dof entry (the bodies'), zero here
        if (phase == CLUSTER_KE) block_reduce_store<3>(ke, S.kePart, tile.slot);
        else if (phase == CLUSTER_PART2) {
            double k2[2] = {ke[0], 0.0};
            block_reduce_store<2>(k2, S.kePart, tile.slot);
        }
    }
}

// positions as the force field reads them, as a hi part and a low part:
// body atoms (and the massless particles after them) at their fp32
// positions in mixed precision (lo = 0), free atoms at hi + lo
template <class Real, class IO = SoaAtoms>
__device__ __forceinline__ void field_pos_parts(const DevSys& S, int i, int s, V3<Real>& hi, V3<Real>& lo) {
    lo = {(Real)0, (Real)0, (Real)0};
    if constexpr (IO::adopted) {
        Q4<Real> p = ld4<Real>(S.ommPosq, s);
        hi = {p.a, p.b, p.c};
        if (sizeof(Real) == 4 && i < S.numFree) {
            const float* c = S.ommPosqCorr + 4 * (size_t)s;
            lo = {(Real)c[0], (Real)c[1], (Real)c[2]};
        }
    } else {
        hi = ld3<Real>(S.pos, S.atomStride, i);
        if (sizeof(Real) == 4 && i < S.numFree) lo = cvt<Real>(ld3<float>(S.posLo, S.atomStride, i));
    }
}
template <class Real, class IO = SoaAtoms> __device__ __forceinline__ V3<double> force_pos(const DevSys& S, int i) {
    V3<Real> hi, lo;
    field_pos_parts<Real, IO>(S, i, IO::at(S, i), hi, lo);
    return cvt<double>(hi) + cvt<double>(lo);
}
// a force into the library's array, or into the adopted fixed-point array
template <class Real, class IO> __device__ __forceinline__ void store_force(const DevSys& S, int at, V3<Real> f) {
    if constexpr (IO::adopted) {
        long long* o = S.ommForce + at;
        const size_t st = (size_t)S.ommStride;
        o[0] = IO::fixed_point((double)f.x);
        o[st] = IO::fixed_point((double)f.y);
        o[2 * st] = IO::fixed_point((double)f.z);
    } else {
        st3<Real>(S.force, S.atomStride, at, f);
    }
}

// ---------------------------------------------------------------------------
// Virtual sites (OpenMM's, placed after part 1 and the constraints,
// ReferenceRigidBodyKernels.cpp:100): two- and three-particle averages and
// out-of-plane sites from their parents' positions; after the forces, each
// parent gathers the force of its sites (the transpose of d r_site /
// d r_parent) in a fixed order, and the sites' forces are cleared.  One lane
// per site or per parent.
// ---------------------------------------------------------------------------
// the local frame of a local-coordinates site: x and y are the x- and
// y-weighted sums of the parents, e_x = x/|x|, e_z = (x × y)/|x × y|,
// e_y = e_z × e_x
struct SiteFrame { V3<double> x, y, ex, ey, ez; double nx, nz; };

template <class Real>
__device__ __forceinline__ SiteFrame site_frame(const DevSys& S, const int* p, const double* w) {
    SiteFrame f;
    V3<double> r0 = force_pos<Real>(S, p[0]), r1 = force_pos<Real>(S, p[1]), r2 = force_pos<Real>(S, p[2]);
    f.x = r0 * w[3] + r1 * w[4] + r2 * w[5];
    f.y = r0 * w[6] + r1 * w[7] + r2 * w[8];
    V3<double> z = cross(f.x, f.y);
    f.nx = sqrt(dot(f.x, f.x));
    f.nz = sqrt(dot(z, z));
    f.ex = f.x * (1.0 / f.nx);
    f.ez = z * (1.0 / f.nz);
    f.ey = cross(f.ez, f.ex);
    return f;
}

template <class Real>
__global__ __launch_bounds__(256) void k_site_positions(const DevSys* __restrict__ sys) {
    const DevSys& S = *sys;
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= S.numSites) return;
    const int* p = S.siteParent + 3 * (size_t)s;
    const double* w = S.siteW + 12 * (size_t)s;
    V3<double> r1 = force_pos<Real>(S, p[0]), r2 = force_pos<Real>(S, p[1]), x;
    const int type = S.siteType[s];
    if (type == SITE_LOCAL_COORDINATES) {
        SiteFrame f = site_frame<Real>(S, p, w);
        V3<double> o = r1 * w[0] + r2 * w[1] + force_pos<Real>(S, p[2]) * w[2];
        x = o + f.ex * w[9] + f.ey * w[10] + f.ez * w[11];
    } else if (type == SITE_TWO_AVERAGE) {
        x = r1 * w[0] + r2 * w[1];
    } else if (type == SITE_THREE_AVERAGE) {
        x = r1 * w[0] + r2 * w[1] + force_pos<Real>(S, p[2]) * w[2];
    } else {
        V3<double> r12 = r2 - r1, r13 = force_pos<Real>(S, p[2]) - r1;
        x = r1 + r12 * w[0] + r13 * w[1] + cross(r12, r13) * w[2];
    }
    store_pos<Real>(S, S.siteAtom[s], x);
}

template <class Real>
__global__ __launch_bounds__(256) void k_site_forces(const DevSys* __restrict__ sys) {
    const DevSys& S = *sys;
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= S.numSiteParents) return;
    const int a = S.parentAtom[g];
    V3<double> f = cvt<double>(ld3<Real>(S.force, S.atomStride, a));
    for (int e = S.parentStart[g]; e < S.parentStart[g + 1]; e++) {
        const int s = S.parentSite[e], role = S.parentRole[e];
        const int* p = S.siteParent + 3 * (size_t)s;
        const double* w = S.siteW + 12 * (size_t)s;
        V3<double> fs = cvt<double>(ld3<Real>(S.force, S.atomStride, S.siteAtom[s]));
        const int type = S.siteType[s];
        if (type == SITE_TWO_AVERAGE || type == SITE_THREE_AVERAGE) {
            f = f + scaled(fs, w[role]);
        } else if (type == SITE_LOCAL_COORDINATES) {
            // ow F + xw Gx + yw Gy, Gx and Gy the transposed derivatives of
            // the site with respect to x and y
            SiteFrame fr = site_frame<Real>(S, p, w);
            auto Jx = [&](V3<double> a) { return (a - fr.ex * dot(fr.ex, a)) * (1.0 / fr.nx); };
            auto Jz = [&](V3<double> a) { return (a - fr.ez * dot(fr.ez, a)) * (1.0 / fr.nz); };
            V3<double> jzexf = Jz(cross(fr.ex, fs)), jzf = Jz(fs);
            V3<double> gx = Jx(fs) * w[9] + (cross(fr.y, jzexf) - Jx(cross(fr.ez, fs))) * w[10] + cross(fr.y, jzf) * w[11];
            V3<double> gy = cross(fr.x, jzexf) * (-w[10]) - cross(fr.x, jzf) * w[11];
            f = f + (fs * w[role] + gx * w[3 + role] + gy * w[6 + role]);
        } else {
            V3<double> r1 = force_pos<Real>(S, p[0]);
            V3<double> r12 = force_pos<Real>(S, p[1]) - r1, r13 = force_pos<Real>(S, p[2]) - r1;
            V3<double> f2 = fs * w[0] + cross(r13, fs) * w[2];
            V3<double> f3 = fs * w[1] + cross(fs, r12) * w[2];
            f = f + (role == 0 ? fs - f2 - f3 : role == 1 ? f2 : f3);
        }
    }
    st3<Real>(S.force, S.atomStride, a, cvt<Real>(f));
}

template <class Real>
__global__ __launch_bounds__(256) void k_site_clear(const DevSys* __restrict__ sys) {
    const DevSys& S = *sys;
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= S.numSites) return;
    st3<Real>(S.force, S.atomStride, S.siteAtom[s], V3<Real>{(Real)0, (Real)0, (Real)0});
}

// ---------------------------------------------------------------------------
// force field: harmonic tether + harmonic bonds, one lane per atom.  Body
// atoms are read at their fp32 positions (as a mixed-precision force field
// reads fp32 coordinates), free atoms at hi + lo; the tether's anchor r0 is
// held at the state precision (fp32 in mixed precision, as a mixed-precision
// force field holds its parameters), so an atom moves 36 bytes: its
// position, r0 and its force.  With ENERGY the tiles' potential-energy
// partials too; a step asks for forces only (calcForcesAndEnergy(true,
// false), ReferenceRigidBodyKernels.cpp:101), so a sequence of steps takes
// the energy at its last evaluation alone.
// ---------------------------------------------------------------------------

// -k dx, rounded (never fused into the sum it goes to, so a force summed in
// registers equals one that went through the force array)
template <class Real> __device__ __forceinline__ V3<Real> tether_force(V3<Real> dx, Real k) {
#pragma clang fp contract(off)
    return {dx.x * (-k), dx.y * (-k), dx.z * (-k)};
}

template <class Real, class IO, bool ENERGY>
__global__ __launch_bounds__(512) void k_forces(const DevSys* __restrict__ systems, const Tile* __restrict__ tiles,
                                                 int numTiles) {
    for (int t = blockIdx.x; t < numTiles; t += gridDim.x) {
        const Tile tile = tiles[t];
        // (a copy: read through the table, the descriptor's fields would be
        // re-read after every store, which may alias it, and each re-read
        // waits for the atom loads in flight)
        const DevSys S = systems[tile.sys];
        double e[1] = {0.0};
        constexpr int U = force_batch<Real, IO>();
        const bool tethered = S.tetherScale != 0.0;
        for (int i0 = threadIdx.x; i0 < tile.count; i0 += U * blockDim.x) {
            int at[U];
            V3<Real> ph[U], pl[U], r0[U];
            Real k[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                if (i0 + u * (int)blockDim.x < tile.count) at[u] = IO::at(S, tile.first + i0 + u * blockDim.x);
            if (tethered) {
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int a = tile.first + i0 + u * blockDim.x;
                    if (i0 + u * (int)blockDim.x < tile.count) {
                        field_pos_parts<Real, IO>(S, a, at[u], ph[u], pl[u]);
                        r0[u] = ld3<Real>(S.r0, S.atomStride, a);
                        k[u] = S.tetherUniform ? (Real)S.tetherK0 : reinterpret_cast<const Real*>(S.tetherK)[a];
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (i0 + u * (int)blockDim.x >= tile.count) break;
                const int a = tile.first + i0 + u * blockDim.x;
                V3<Real> f = {(Real)0, (Real)0, (Real)0};
                if (tethered) {
                    V3<Real> dx = (ph[u] - r0[u]) + pl[u];
                    f = tether_force(dx, k[u]);
                    if (ENERGY) {
                        V3<double> dd = cvt<double>(dx);
                        e[0] += 0.5 * (double)k[u] * dot(dd, dd);
                    }
                }
                if (S.bondStart) {
                    int e0 = S.bondStart[a], e1 = S.bondStart[a + 1];
                    if (e0 < e1) {
                        V3<double> pa = force_pos<Real, IO>(S, a);
                        V3<double> fd = cvt<double>(f);
                        for (int b = e0; b < e1; b++) {
                            V3<double> dr = force_pos<Real, IO>(S, S.bondOther[b]) - pa;
                            double r = sqrt(dot(dr, dr));
                            double ext = r - S.bondLen[b];
                            fd = fd + dr * (S.bondK[b] * ext / r);
                            if (ENERGY) e[0] += 0.25 * S.bondK[b] * ext * ext;
                        }
                        f = cvt<Real>(fd);
                    }
                }
                store_force<Real, IO>(S, at[u], f);
            }
        }
        if (ENERGY) block_reduce_store<1>(e, S.pePart, tile.slot);
    }
}

// ---------------------------------------------------------------------------
// Steps of systems whose force on an atom depends on that atom alone (no
// bonds: the tether, or no force), or by way of a virtual site on its own body.
// A body's interior step boundaries then need nothing from other bodies, and a
// constraint cluster's nothing from other atoms, so one launch carries
// each body (each free atom) through `boundaries` x [forces, fused pass] with
// its state in registers and its atoms' coordinates and anchors in LDS:
// positions, forces and body state go through memory once per launch instead
// of once per step.  The arithmetic and every rounding to the state precision
// are those of k_part1, k_forces and k_fused (the fused operations whose
// choice the compiler makes by context are written out: step_rot, step_apply,
// to_body, kicked, the exact rotation), so results are the same bit for bit as
// part 1, then [forces, fused pass], gives.
// FIRST: a part 1 comes before the boundaries; LAST: the atom positions are
// written at the end (a launch that continues another reads only the body
// state).
//
// What bounds it: VALU issue (NO-SQUISH: 41 turns of 24 instructions in the
// ~1300 of a body's step; FP64 latency with the exact rotation), no longer
// HBM.  Per step, k_fused + k_forces -> k_steps: 1M waters, NO-SQUISH 10,
// 58.2 -> 24.1 us; 20k waters 9.9 -> 2.8 us; the heterogeneous mix (200k
// bodies, 500k free atoms, exact) 32.5 -> 8.3 us; 512 waters in FP64, exact,
// 9.3 -> 2.9 us.  One wave per workgroup: tiles end apart, and the launch
// fills the SIMDs evenly.  kStepsPerLaunch: 16, 64, 256 and 2048 boundaries
// per launch ran the 1M waters at 25.7, 24.1, 24.6 and 25.1 us and the
// heterogeneous mix at 9.0, 8.3, 8.2 and 8.3; 64 leaves other streams a slot
// every few ms (a server's set-ups: 29 against 31 ms for a backlog with 2048).
//
// Sites and clusters (10k four-site waters and 2000 triangles, per step): six
// kernels, 31.6 us -> bodies and sites 4.1 us beside clusters 7.0 us, the latter
// bound by the serial FP64 sweeps of their 32 waves (fewer clusters per wave, so
// that a wave waits for fewer sweeps, were slower: 8.0 with 16, 13.7 with 2).  A body with
// sites takes its forces atom by atom in a loop of its own (site_sums), in an
// instance that systems without sites do not run.
//
// LDS: each lane keeps its own atoms' {d, r0, k}, 7 Reals per atom, at an odd
// stride of Reals, so the lanes of a wave hit different banks; a lane reads
// only what it wrote, so there is no barrier.  One copy of the rotation
// serves every body size (the sizes differ in the sums only): with one per
// size the exact kernel needed 256 + 14 registers and ran one wave per SIMD.
// ---------------------------------------------------------------------------
enum : int { STEPS_FIRST = 1, STEPS_LAST = 2 };

// adds one tethered atom's force and torque to F and tau (a: its {d, r0, k})
template <class Real, bool YFIRST, bool SMALL, class IO>
__device__ __forceinline__ void add_tethered(const Real* a, bool uniform, Real k0, const Rot<Real>& R, V3<double> rc,
                                             bool xfirst, V3<double>& F, V3<double>& tau) {
    const V3<Real> d = {a[0], a[1], a[2]};
    V3<double> dl = cvt<double>(step_apply<YFIRST>(R, d));
    V3<Real> x = cvt<Real>(rc + (SMALL && xfirst ? cvt<double>(place_apply<true>(R, d)) : dl));
    V3<double> f = cvt<double>(IO::held_force(tether_force(x - V3<Real>{a[3], a[4], a[5]}, uniform ? k0 : a[6])));
    F = F + f;
    tau = tau + cross(dl, f);
}

// F and tau of one body's (or one lane's share of its) atoms at st, in the
// order and with the rounding of body_sums (N: the body's atoms if one lane
// has them all)
template <class Real, bool EXACT, class IO>
__device__ __forceinline__ void tethered_sums(const Real* st, int N, int per, bool uniform, Real k0,
                                              const Rot<Real>& R, V3<double> rc, bool xfirst, V3<double>& F,
                                              V3<double>& tau) {
    auto fixed = [&](auto NC) {
#pragma unroll
        for (int u = 0; u < NC; u++)
            add_tethered<Real, true, (!EXACT && decltype(NC)::value <= 4), IO>(st + 7 * u, uniform, k0, R, rc, xfirst,
                                                                               F, tau);
    };
    switch (N) {
    case 2: fixed(std::integral_constant<int, 2>{}); break;
    case 3: fixed(std::integral_constant<int, 3>{}); break;
    case 4: fixed(std::integral_constant<int, 4>{}); break;
    case 6: fixed(std::integral_constant<int, 6>{}); break;
    default:
        for (int u0 = 0; u0 < per; u0 += STRIDED_BATCH) {
            add_tethered<Real, true, false, IO>(st + 7 * u0, uniform, k0, R, rc, false, F, tau);
            const int end = per < u0 + STRIDED_BATCH ? per : u0 + STRIDED_BATCH;
            for (int u = u0 + 1; u < end; u++)
                add_tethered<Real, false, false, IO>(st + 7 * u, uniform, k0, R, rc, false, F, tau);
        }
    }
}

// A body's virtual sites, kSiteReals of Real each after its atoms: the weights
// (FP64), anchor and spring constant, the parents' places in the body, and the
// force on the site while a step's sums are taken.
constexpr int kNoParent = 1023;
template <class Real> struct SiteRecord {
    Real* a;
    static constexpr int W = sizeof(double) / sizeof(Real);   // Reals per FP64 value
    __device__ __forceinline__ void set_weight(int i, double w) { __builtin_memcpy(a + W * i, &w, sizeof(w)); }
    __device__ __forceinline__ double weight(int i) const {
        double w;
        __builtin_memcpy(&w, a + W * i, sizeof(w));
        return w;
    }
    __device__ __forceinline__ V3<Real>& r0() const { return *reinterpret_cast<V3<Real>*>(a + 3 * W); }
    __device__ __forceinline__ Real& k() const { return a[3 * W + 3]; }
    __device__ __forceinline__ void set_parents(int p) { __builtin_memcpy(a + 3 * W + 4, &p, sizeof(p)); }
    __device__ __forceinline__ int parents() const {
        int p;
        __builtin_memcpy(&p, a + 3 * W + 4, sizeof(p));
        return p;
    }
    __device__ __forceinline__ V3<Real>& force() const { return *reinterpret_cast<V3<Real>*>(a + 3 * W + 5); }
};

template <class Real>
__device__ __forceinline__ void load_site(const DevSys& S, SiteRecord<Real> r, int s, int atom0) {
    const int a = S.siteAtom[s], two = S.siteType[s] == SITE_TWO_AVERAGE;
    const int* p = S.siteParent + 3 * (size_t)s;
    const double* w = S.siteW + 12 * (size_t)s;
    for (int i = 0; i < 3; i++) r.set_weight(i, w[i]);
    r.r0() = ld3<Real>(S.r0, S.atomStride, a);
    r.k() = S.tetherUniform ? (Real)S.tetherK0 : reinterpret_cast<const Real*>(S.tetherK)[a];
    r.set_parents((p[0] - atom0) | (p[1] - atom0) << 10 | (two ? kNoParent : p[2] - atom0) << 20);
}

// F and tau of one lane's whole body with sites: as tethered_sums, each force
// with its share of the sites' forces added and rounded as k_site_forces does
template <class Real, bool EXACT>
__device__ __forceinline__ void site_sums(const Real* st, Real* sites, int numSites, int N, bool xfirst, bool uniform,
                                          Real k0, const Rot<Real>& R, V3<double> rc, V3<double>& F,
                                          V3<double>& tau) {
    const bool fixed = N == 2 || N == 3 || N == 4 || N == 6;
    auto offset = [&](int j) {
        const V3<Real> d = {st[7 * j], st[7 * j + 1], st[7 * j + 2]};
        return fixed ? step_apply<true>(R, d) : strided_apply(R, d, j);
    };
    auto place = [&](int j) {
        const V3<Real> d = {st[7 * j], st[7 * j + 1], st[7 * j + 2]};
        return cvt<Real>(rc + cvt<double>(xfirst ? place_apply<true>(R, d) : offset(j)));
    };
    for (int s = 0; s < numSites; s++) {
        const SiteRecord<Real> r{sites + kSiteReals * s};
        const int p = r.parents(), p2 = p >> 20 & 1023;
        const double w0 = r.weight(0), w1 = r.weight(1);
        const V3<double> x0 = cvt<double>(place(p & 1023)), x1 = cvt<double>(place(p >> 10 & 1023));
        V3<double> x = {fma(x0.x, w0, x1.x * w1), fma(x0.y, w0, x1.y * w1), fma(x0.z, w0, x1.z * w1)};
        if (p2 != kNoParent) {
            const double w2 = r.weight(2);
            const V3<double> x2 = cvt<double>(place(p2));
            x = {fma(x2.x, w2, x.x), fma(x2.y, w2, x.y), fma(x2.z, w2, x.z)};
        }
        r.force() = tether_force(cvt<Real>(x) - r.r0(), r.k());
    }
    for (int j = 0; j < N; j++) {
        const Real* a = st + 7 * j;
        V3<double> f = cvt<double>(tether_force(place(j) - V3<Real>{a[3], a[4], a[5]}, uniform ? k0 : a[6]));
        for (int s = 0; s < numSites; s++) {
            const SiteRecord<Real> r{sites + kSiteReals * s};
            const int p = r.parents();
            const V3<double> fs = cvt<double>(r.force());
            for (int i = 0; i < 3; i++)
                if ((p >> 10 * i & 1023) == j) f = f + scaled(fs, r.weight(i));
        }
        f = cvt<double>(cvt<Real>(f));
        const V3<double> dl = cvt<double>(offset(j));
        F = F + f;
        tau = tau + cross(dl, f);
    }
}

template <class Real, bool EXACT, class IO, bool SITES>
__device__ __forceinline__ void steps_bodies(const DevSys& S, const Tile& tile, int boundaries, int flags,
                                             Real* stash) {
    const int N = tile.N, lanes = tile.lanes;
    const int b = threadIdx.x >> lane_shift(lanes);
    const int sub = threadIdx.x & (lanes - 1);
    if (b >= tile.count) return;
    const int k = tile.first + b;
    const int atom0 = tile.atomFirst + b * N;
    const Shape sh = body_shape(S, tile, k, atom0, N);
    const int perMax = (N + lanes - 1) / lanes;
    const int per = (N - sub + lanes - 1) / lanes;
    Real* st = stash + (size_t)threadIdx.x * ((7 * perMax + (SITES ? kSiteReals * S.maxBodySites : 0)) | 1);
    Real* sites = st + 7 * perMax;
    int numSites = 0;
    if constexpr (SITES) {
        if (S.maxBodySites > 0) {
            const int first = S.bodySiteStart[k];
            numSites = S.bodySiteStart[k + 1] - first;
            for (int s = 0; s < numSites; s++)
                load_site<Real>(S, SiteRecord<Real>{sites + kSiteReals * s}, S.bodySites[first + s], atom0);
        }
    }
    const bool tethered = S.tetherScale != 0.0, uniform = S.tetherUniform != 0;
    const Real k0 = (Real)S.tetherK0;
    for (int u = 0; u < per; u++) {
        const int j = sub + u * lanes;
        V3<Real> d = ld3<Real>(S.d, S.dStride, sh.row + j);
        V3<Real> r0 = ld3<Real>(S.r0, S.atomStride, atom0 + j);
        Real* a = st + 7 * u;
        a[0] = d.x; a[1] = d.y; a[2] = d.z;
        a[3] = r0.x; a[4] = r0.y; a[5] = r0.z;
        a[6] = uniform ? k0 : reinterpret_cast<const Real*>(S.tetherK)[atom0 + j];
    }
    Body<Real> B = load_body<Real>(S, k, sh.ks);
    V3<double> rc = load_rcm<Real>(S, k);
    const bool small = small_body(S, N, lanes);
    const int first = (flags & STEPS_FIRST) ? -1 : 0;
    // whether step s's positions have row 0's x products rounded: those of
    // small bodies, where the fused pass places them, and of 4 atoms where
    // part 1 does (before step 0), which places 2 and 3 the other way
    auto xfirst = [&](int s) { return small && (N == 4 || s > 0 || !(flags & STEPS_FIRST)); };
    for (int s = first; s < boundaries; s++) {
        if (s >= 0) {
            Rot<Real> R = step_rot(B.q);
            V3<double> F = {0.0, 0.0, 0.0}, tau = {0.0, 0.0, 0.0};
            if (SITES && tethered && numSites > 0)
                site_sums<Real, EXACT>(st, sites, numSites, N, xfirst(s), uniform, k0, R, rc, F, tau);
            else if (tethered)
                tethered_sums<Real, EXACT, IO>(st, lanes == 1 ? N : 0, per, uniform, k0, R, rc, xfirst(s), F, tau);
            if (lanes > 1) {
                F = {xor_sum(F.x, lanes), xor_sum(F.y, lanes), xor_sum(F.z, lanes)};
                tau = {xor_sum(tau.x, lanes), xor_sum(tau.y, lanes), xor_sum(tau.z, lanes)};
            }
            fused_kicks<Real>(S, B, R, F, tau, small);
        }
        drift_and_rotate<Real, EXACT>(S, B, rc);
    }
    if (sub == 0) store_body<Real>(S, k, B, rc);
    if (flags & STEPS_LAST) {
        Rot<Real> R = step_rot(B.q);
        const bool fixed = lanes == 1 && (N == 2 || N == 3 || N == 4 || N == 6);
        for (int u = 0; u < per; u++) {
            const V3<Real> d = {st[7 * u], st[7 * u + 1], st[7 * u + 2]};
            const V3<Real> dl = !fixed                ? strided_apply(R, d, u)
                                : xfirst(boundaries) ? place_apply<true>(R, d)
                                                     : step_apply<true>(R, d);
            const int at = IO::at(S, atom0 + sub + u * lanes);
            IO::template set_body_pos_at<Real>(S, at, rc + cvt<double>(dl));
        }
    }
}

template <class Real, class IO>
__device__ __forceinline__ void steps_free(const DevSys& S, const Tile& tile, int boundaries, int flags) {
    const Real halfDt = (Real)(0.5 * S.dt);
    const bool tethered = S.tetherScale != 0.0, uniform = S.tetherUniform != 0;
    for (int i = threadIdx.x; i < tile.count; i += blockDim.x) {
        const int a = tile.first + i;
        V3<Real> v = IO::template vel<Real>(S, a);
        const Real invm = reinterpret_cast<const Real*>(S.freeInvM)[a];
        const V3<Real> r0 = ld3<Real>(S.r0, S.atomStride, a);
        const Real k = uniform ? (Real)S.tetherK0 : reinterpret_cast<const Real*>(S.tetherK)[a];
        V3<double> r = IO::template pos<Real>(S, a);
        // the stored position: hi + lo in mixed precision
        V3<Real> hi = cvt<Real>(r), lo = {(Real)0, (Real)0, (Real)0};
        auto split = [&] {
            hi = cvt<Real>(r);
            if (sizeof(Real) == 4) {
                lo = cvt<Real>(r - cvt<double>(hi));
                r = cvt<double>(hi) + cvt<double>(lo);
            }
        };
        split();
        if (flags & STEPS_FIRST) {
            V3<Real> f = IO::template force<Real>(S, a);
            v = v + f * invm * halfDt;
            r = r + cvt<double>(v) * S.dt;
            split();
        }
        for (int s = 0; s < boundaries; s++) {
            V3<Real> f = {(Real)0, (Real)0, (Real)0};
            if (tethered) f = IO::held_force(tether_force((hi - r0) + lo, k));
            v = v + f * invm * halfDt;     // end of step n
            v = v + f * invm * halfDt;     // start of step n+1
            r = r + cvt<double>(v) * S.dt;
            split();
        }
        IO::template set_vel<Real>(S, a, v);
        IO::template set_pos<Real>(S, a, r);
    }
}

// the same for one constraint cluster of NA atoms
template <class Real, int NA>
__device__ __forceinline__ void steps_cluster(const DevSys& S, int c, int boundaries, int flags) {
    SmallCluster<Real, NA> K;
    K.load(S, c);
    const bool tethered = S.tetherScale != 0.0;
    Four<V3<Real>> r0, f;
    Four<Real> k;
    static_for<NA>([&](auto J) {
        constexpr int j = J;
        const int a = K.atom.template at<j>();
        r0.template at<j>() = ld3<Real>(S.r0, S.atomStride, a);
        k.template at<j>() = S.tetherUniform ? (Real)S.tetherK0 : reinterpret_cast<const Real*>(S.tetherK)[a];
    });
    // the force at the stored position (hi + lo in mixed precision), to which
    // the position is rounded
    auto forces = [&] {
        static_for<NA>([&](auto J) {
            constexpr int j = J;
            V3<double>& r = K.r.template at<j>();
            V3<Real> hi = cvt<Real>(r), lo = {(Real)0, (Real)0, (Real)0};
            if (sizeof(Real) == 4) {
                lo = cvt<Real>(r - cvt<double>(hi));
                r = cvt<double>(hi) + cvt<double>(lo);
            }
            f.template at<j>() = tethered ? tether_force((hi - r0.template at<j>()) + lo, k.template at<j>())
                                          : V3<Real>{(Real)0, (Real)0, (Real)0};
        });
    };
    unsigned failed = 0;
    if (flags & STEPS_FIRST) {
        f = K.stored_forces(S);
        failed += !K.begin_step(S, f);
    }
    for (int s = 0; s < boundaries; s++) {
        forces();
        const bool ended = K.end_step(S, f), begun = K.begin_step(S, f);
        failed += !(ended && begun);
    }
    K.store_positions(S);
    K.store_velocities(S);
    if (failed) atomicAdd(S.constraintFail, failed);
}

template <class Real, bool EXACT, class IO, bool SITES>
__global__ __launch_bounds__(kStepsBlock) __attribute__((amdgpu_waves_per_eu(2))) void k_steps(const DevSys* __restrict__ systems,
                                                              const Tile* __restrict__ tiles, int numTiles,
                                                              int boundaries, int flags) {
    extern __shared__ double stash_memory[];
    Real* stash = reinterpret_cast<Real*>(stash_memory);
    for (int t = blockIdx.x; t < numTiles; t += gridDim.x) {
        const Tile tile = tiles[t];
        const DevSys& S = systems[tile.sys];
        if (tile.kind == TILE_FREE) {
            steps_free<Real, IO>(S, tile, boundaries, flags);
            continue;
        }
        steps_bodies<Real, EXACT, IO, SITES>(S, tile, boundaries, flags, stash);
    }
}

// constraint clusters of NA = 2, 3 or 4 atoms, one lane each
template <class Real, int NA>
__global__ __launch_bounds__(kStepsBlock) void k_cluster_steps(const DevSys* __restrict__ systems,
                                                               const Tile* __restrict__ tiles, int boundaries,
                                                               int flags) {
    const Tile tile = tiles[blockIdx.x];
    const DevSys& S = systems[tile.sys];
    if ((int)threadIdx.x < tile.count) steps_cluster<Real, NA>(S, tile.first + threadIdx.x, boundaries, flags);
}

// bodies, free atoms and clusters of 2 and 3 atoms side by side, the clusters,
// which take longest, first
template <class Real, bool EXACT>
__global__ __launch_bounds__(kStepsBlock) __attribute__((amdgpu_waves_per_eu(2))) void k_steps_mixed(
    const DevSys* __restrict__ systems, const Tile* __restrict__ tiles, const Tile* __restrict__ clusterTiles,
    int numClusterTiles, int boundaries, int flags) {
    extern __shared__ double stash_memory[];
    const int t = (int)blockIdx.x - numClusterTiles;
    const Tile tile = t < 0 ? clusterTiles[blockIdx.x] : tiles[t];
    const DevSys& S = systems[tile.sys];
    if (tile.kind == TILE_CLUSTERS) {
        if ((int)threadIdx.x >= tile.count) return;
        if (tile.N == 2) steps_cluster<Real, 2>(S, tile.first + threadIdx.x, boundaries, flags);
        else steps_cluster<Real, 3>(S, tile.first + threadIdx.x, boundaries, flags);
    } else if (tile.kind == TILE_FREE) {
        steps_free<Real, SoaAtoms>(S, tile, boundaries, flags);
    } else {
        steps_bodies<Real, EXACT, SoaAtoms, true>(S, tile, boundaries, flags, reinterpret_cast<Real*>(stash_memory));
    }
}

// deterministic sum of the 4-double partials of each system; one block per
// system.  nslots: their count per system, or null for `count` (one system).
// `out` may be pinned host memory: a context's energies are written there by
// the kernel, so a query is one launch and one wait (28 us with the count
// copied up and the sum copied down, 13 without).
__global__ __launch_bounds__(256) void k_reduce(const DevSys* __restrict__ systems, const int* __restrict__ nslots,
                                                 int count, int which, double* __restrict__ out) {
    const DevSys& S = systems[blockIdx.x];
    const double* part = which == 0 ? S.kePart : which == 1 ? S.pePart : which == 2 ? S.refKePart : S.refPePart;
    int n = nslots ? nslots[blockIdx.x] : count;
    __shared__ double red[256][4];
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int s = threadIdx.x; s < n; s += blockDim.x)
        for (int c = 0; c < 4; c++) acc[c] += part[4 * (size_t)s + c];
    for (int c = 0; c < 4; c++) red[threadIdx.x][c] = acc[c];
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int c = 0; c < 4; c++) red[threadIdx.x][c] += red[threadIdx.x + w][c];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int c = 0; c < 4; c++) out[4 * (size_t)blockIdx.x + c] = red[0][c];
}

__global__ void k_copy(const float4* __restrict__ src, float4* __restrict__ dst, size_t n) {
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static int grid_for(int numTiles, int maxBlocks) {
    if (numTiles <= 0) return 0;
    return maxBlocks > 0 && maxBlocks < numTiles ? maxBlocks : numTiles;
}

// Timing of the step kernels: with events set by set_step_kernel_events
// (per thread), the next step kernel is launched with them attached to its
// dispatch (hipExtLaunchKernelGGL), so they record its own start and end;
// both are then cleared.  Without them, a plain launch.
namespace {
thread_local hipEvent_t t_kernelStart = nullptr, t_kernelStop = nullptr;

template <class... KArgs, class... Args>
void step_kernel_lds(void (*kernel)(KArgs...), int grid, int block, size_t lds, hipStream_t stream, Args... args) {
    if (t_kernelStart) {
        hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(block), lds, stream, t_kernelStart, t_kernelStop, 0, args...);
        t_kernelStart = t_kernelStop = nullptr;
    } else {
        kernel<<<grid, block, lds, stream>>>(args...);
    }
}
template <class... KArgs, class... Args>
void step_kernel(void (*kernel)(KArgs...), int grid, int block, hipStream_t stream, Args... args) {
    step_kernel_lds(kernel, grid, block, 0, stream, args...);
}
}  // namespace

void set_step_kernel_events(hipEvent_t start, hipEvent_t stop) {
    t_kernelStart = start;
    t_kernelStop = stop;
}

bool clear_step_kernel_events() {
    const bool pending = t_kernelStart != nullptr;
    t_kernelStart = t_kernelStop = nullptr;
    return pending;
}

// the step kernels for the atom layout (library arrays or adopted arrays),
// state precision and rotation kind
template <class IO>
static void part1_for(int precision, int rotationMode, int grid, int block, hipStream_t stream,
                      const DevSys* systems, const Tile* tiles, int numTiles) {
    if (precision == 0) {
        if (rotationMode == 0) step_kernel(k_part1<float, true, IO>, grid, block, stream, systems, tiles, numTiles);
        else step_kernel(k_part1<float, false, IO>, grid, block, stream, systems, tiles, numTiles);
    } else {
        if (rotationMode == 0) step_kernel(k_part1<double, true, IO>, grid, block, stream, systems, tiles, numTiles);
        else step_kernel(k_part1<double, false, IO>, grid, block, stream, systems, tiles, numTiles);
    }
}
template <class IO>
static void fused_for(int precision, int rotationMode, int grid, int block, hipStream_t stream,
                      const DevSys* systems, const Tile* tiles, int numTiles) {
    if (precision == 0) {
        if (rotationMode == 0) step_kernel(k_fused<float, true, IO>, grid, block, stream, systems, tiles, numTiles);
        else step_kernel(k_fused<float, false, IO>, grid, block, stream, systems, tiles, numTiles);
    } else {
        if (rotationMode == 0) step_kernel(k_fused<double, true, IO>, grid, block, stream, systems, tiles, numTiles);
        else step_kernel(k_fused<double, false, IO>, grid, block, stream, systems, tiles, numTiles);
    }
}

hipError_t launch_part1(int precision, int rotationMode, const DevSys* systems, const Tile* tiles, int numTiles,
                        int block, int maxBlocks, hipStream_t stream, int adopted) {
    int grid = grid_for(numTiles, maxBlocks);
    if (grid == 0) return hipSuccess;
    if (adopted) part1_for<AdoptedAtoms>(precision, rotationMode, grid, block, stream, systems, tiles, numTiles);
    else part1_for<SoaAtoms>(precision, rotationMode, grid, block, stream, systems, tiles, numTiles);
    return hipGetLastError();
}

hipError_t launch_fused(int precision, int rotationMode, const DevSys* systems, const Tile* tiles, int numTiles,
                        int block, int maxBlocks, hipStream_t stream, int adopted) {
    int grid = grid_for(numTiles, maxBlocks);
    if (grid == 0) return hipSuccess;
    if (adopted) fused_for<AdoptedAtoms>(precision, rotationMode, grid, block, stream, systems, tiles, numTiles);
    else fused_for<SoaAtoms>(precision, rotationMode, grid, block, stream, systems, tiles, numTiles);
    return hipGetLastError();
}

// The free-atom tiles' kinetic-energy partials again, from the adopted
// velocities as they are now (after the caller's velocity constraints), into
// the slots part 2 filled; body tiles keep theirs.
template <class Real>
__global__ __launch_bounds__(512) void k_free_ke(const DevSys* __restrict__ systems, const Tile* __restrict__ tiles,
                                                  int numTiles) {
    for (int t = blockIdx.x; t < numTiles; t += gridDim.x) {
        const Tile tile = tiles[t];
        if (tile.kind != TILE_FREE) continue;
        const DevSys& S = systems[tile.sys];
        double ke[2] = {0.0, 0.0};
        for (int i = threadIdx.x; i < tile.count; i += blockDim.x) {
            const int a = tile.first + i;
            V3<double> vd = cvt<double>(AdoptedAtoms::vel<Real>(S, a));
            ke[0] += dot(vd, vd) / (double)reinterpret_cast<const Real*>(S.freeInvM)[a];
        }
        block_reduce_store<2>(ke, S.kePart, tile.slot);
    }
}

hipError_t launch_free_ke(int precision, const DevSys* systems, const Tile* tiles, int numTiles, int block,
                          hipStream_t stream) {
    if (numTiles <= 0) return hipSuccess;
    if (precision == 0) k_free_ke<float><<<numTiles, block, 0, stream>>>(systems, tiles, numTiles);
    else k_free_ke<double><<<numTiles, block, 0, stream>>>(systems, tiles, numTiles);
    return hipGetLastError();
}

hipError_t launch_free_delta(int precision, const DevSys* sys, int numFree, double* posDelta, hipStream_t stream) {
    if (numFree <= 0) return hipSuccess;
    const int grid = (numFree + 255) / 256;
    if (precision == 0) k_free_delta<float><<<grid, 256, 0, stream>>>(sys, posDelta);
    else k_free_delta<double><<<grid, 256, 0, stream>>>(sys, posDelta);
    return hipGetLastError();
}

hipError_t launch_part2(int precision, const DevSys* systems, const Tile* tiles, int numTiles, int block,
                        int maxBlocks, hipStream_t stream, int adopted) {
    int grid = grid_for(numTiles, maxBlocks);
    if (grid == 0) return hipSuccess;
    if (precision == 0) {
        if (adopted) step_kernel(k_part2<float, AdoptedAtoms>, grid, block, stream, systems, tiles, numTiles);
        else step_kernel(k_part2<float, SoaAtoms>, grid, block, stream, systems, tiles, numTiles);
    } else {
        if (adopted) step_kernel(k_part2<double, AdoptedAtoms>, grid, block, stream, systems, tiles, numTiles);
        else step_kernel(k_part2<double, SoaAtoms>, grid, block, stream, systems, tiles, numTiles);
    }
    return hipGetLastError();
}

template <class Real>
static void launch_cluster_classes(const DevSys* systems, const Tile* tiles, const int* counts, int phase, int block,
                                   hipStream_t stream) {
    if (counts[0]) k_clusters<Real, 2><<<counts[0], block, 0, stream>>>(systems, tiles, counts[0], phase);
    tiles += counts[0];
    if (counts[1]) k_clusters<Real, 3><<<counts[1], block, 0, stream>>>(systems, tiles, counts[1], phase);
    tiles += counts[1];
    if (counts[2]) k_clusters<Real, 4><<<counts[2], block, 0, stream>>>(systems, tiles, counts[2], phase);
    tiles += counts[2];
    if (counts[3])
        k_clusters<Real, CLUSTER_MAX_ATOMS><<<counts[3], block, 0, stream>>>(systems, tiles, counts[3], phase);
}

hipError_t launch_clusters(int precision, const DevSys* systems, const Tile* tiles, const int* counts, int phase,
                           int block, hipStream_t stream) {
    if (block > 256) return hipErrorInvalidValue;
    for (int i = 0; i < 4; i++)
        if (counts[i] < 0) return hipErrorInvalidValue;
    if (precision == 0) launch_cluster_classes<float>(systems, tiles, counts, phase, block, stream);
    else launch_cluster_classes<double>(systems, tiles, counts, phase, block, stream);
    return hipGetLastError();
}

hipError_t launch_site_positions(int precision, const DevSys* sys, int numSites, hipStream_t stream) {
    if (numSites <= 0) return hipSuccess;
    const int grid = (numSites + 255) / 256;
    if (precision == 0) k_site_positions<float><<<grid, 256, 0, stream>>>(sys);
    else k_site_positions<double><<<grid, 256, 0, stream>>>(sys);
    return hipGetLastError();
}

hipError_t launch_site_forces(int precision, const DevSys* sys, int numSites, int numParents, hipStream_t stream) {
    if (numSites <= 0) return hipSuccess;
    const int gp = (numParents + 255) / 256, gs = (numSites + 255) / 256;
    if (precision == 0) {
        if (gp) k_site_forces<float><<<gp, 256, 0, stream>>>(sys);
        k_site_clear<float><<<gs, 256, 0, stream>>>(sys);
    } else {
        if (gp) k_site_forces<double><<<gp, 256, 0, stream>>>(sys);
        k_site_clear<double><<<gs, 256, 0, stream>>>(sys);
    }
    return hipGetLastError();
}

template <class Real, bool EXACT>
static void refine_begin_for(int adopted, int grid, int block, hipStream_t stream, const DevSys* systems,
                             const Tile* tiles, int numTiles, int folded) {
    if (adopted) k_refine_begin<Real, EXACT, AdoptedAtoms><<<grid, block, 0, stream>>>(systems, tiles, numTiles, folded);
    else k_refine_begin<Real, EXACT, SoaAtoms><<<grid, block, 0, stream>>>(systems, tiles, numTiles, folded);
}

hipError_t launch_refine_begin(int precision, int rotationMode, const DevSys* systems, const Tile* tiles,
                               int numTiles, int folded, int block, int maxBlocks, hipStream_t stream, int adopted) {
    int grid = grid_for(numTiles, maxBlocks);
    if (grid == 0) return hipSuccess;
    if (precision == 0) {
        if (rotationMode == 0) refine_begin_for<float, true>(adopted, grid, block, stream, systems, tiles, numTiles, folded);
        else refine_begin_for<float, false>(adopted, grid, block, stream, systems, tiles, numTiles, folded);
    } else {
        if (rotationMode == 0) refine_begin_for<double, true>(adopted, grid, block, stream, systems, tiles, numTiles, folded);
        else refine_begin_for<double, false>(adopted, grid, block, stream, systems, tiles, numTiles, folded);
    }
    return hipGetLastError();
}

template <class Real, bool EXACT>
static void refine_end_for(int adopted, int grid, int block, hipStream_t stream, const DevSys* systems,
                           const Tile* tiles, int numTiles) {
    if (adopted) k_refine_end<Real, EXACT, AdoptedAtoms><<<grid, block, 0, stream>>>(systems, tiles, numTiles);
    else k_refine_end<Real, EXACT, SoaAtoms><<<grid, block, 0, stream>>>(systems, tiles, numTiles);
}

hipError_t launch_refine_end(int precision, int rotationMode, const DevSys* systems, const Tile* tiles, int numTiles,
                             int block, int maxBlocks, hipStream_t stream, int adopted) {
    int grid = grid_for(numTiles, maxBlocks);
    if (grid == 0) return hipSuccess;
    if (precision == 0) {
        if (rotationMode == 0) refine_end_for<float, true>(adopted, grid, block, stream, systems, tiles, numTiles);
        else refine_end_for<float, false>(adopted, grid, block, stream, systems, tiles, numTiles);
    } else {
        if (rotationMode == 0) refine_end_for<double, true>(adopted, grid, block, stream, systems, tiles, numTiles);
        else refine_end_for<double, false>(adopted, grid, block, stream, systems, tiles, numTiles);
    }
    return hipGetLastError();
}

hipError_t launch_refine_pe(int precision, const DevSys* systems, const Tile* tiles, int numTiles, int block,
                            int maxBlocks, hipStream_t stream, int adopted) {
    int grid = grid_for(numTiles, maxBlocks);
    if (grid == 0) return hipSuccess;
    if (precision == 0) {
        if (adopted) k_refine_pe<float, AdoptedAtoms><<<grid, block, 0, stream>>>(systems, tiles, numTiles);
        else k_refine_pe<float, SoaAtoms><<<grid, block, 0, stream>>>(systems, tiles, numTiles);
    } else {
        if (adopted) k_refine_pe<double, AdoptedAtoms><<<grid, block, 0, stream>>>(systems, tiles, numTiles);
        else k_refine_pe<double, SoaAtoms><<<grid, block, 0, stream>>>(systems, tiles, numTiles);
    }
    return hipGetLastError();
}

template <class Real, class IO>
static void forces_for(bool energy, int grid, int block, hipStream_t stream, const DevSys* systems, const Tile* tiles,
                       int numTiles) {
    if (energy) step_kernel(k_forces<Real, IO, true>, grid, block, stream, systems, tiles, numTiles);
    else step_kernel(k_forces<Real, IO, false>, grid, block, stream, systems, tiles, numTiles);
}

hipError_t launch_forces(int precision, const DevSys* systems, const Tile* tiles, int numTiles, int block,
                         int maxBlocks, hipStream_t stream, int adopted, int energy) {
    int grid = grid_for(numTiles, maxBlocks);
    if (grid == 0) return hipSuccess;
    if (precision == 0) {
        if (adopted) forces_for<float, AdoptedAtoms>(energy, grid, block, stream, systems, tiles, numTiles);
        else forces_for<float, SoaAtoms>(energy, grid, block, stream, systems, tiles, numTiles);
    } else {
        if (adopted) forces_for<double, AdoptedAtoms>(energy, grid, block, stream, systems, tiles, numTiles);
        else forces_for<double, SoaAtoms>(energy, grid, block, stream, systems, tiles, numTiles);
    }
    return hipGetLastError();
}

template <class IO, bool SITES>
static void steps_for(int precision, int rotationMode, int grid, size_t lds, hipStream_t stream,
                      const DevSys* systems, const Tile* tiles, int numTiles, int boundaries, int flags) {
    auto go = [&](auto kernel) {
        step_kernel_lds(kernel, grid, kStepsBlock, lds, stream, systems, tiles, numTiles, boundaries, flags);
    };
    if (precision == 0) {
        if (rotationMode == 0) go(k_steps<float, true, IO, SITES>);
        else go(k_steps<float, false, IO, SITES>);
    } else {
        if (rotationMode == 0) go(k_steps<double, true, IO, SITES>);
        else go(k_steps<double, false, IO, SITES>);
    }
}

size_t steps_lds_bytes(int precision, int atomsPerLane, int sitesPerLane) {
    const size_t reals = 7 * (size_t)atomsPerLane + (size_t)kSiteReals * sitesPerLane;
    return (size_t)kStepsBlock * (reals | 1) * (precision == 0 ? sizeof(float) : sizeof(double));
}

// One-wave workgroups that a CU's LDS holds, of `lds` bytes each.
static int waves_by_lds(size_t lds) { return (int)((size_t(160) << 10) / lds); }

// Every workgroup of a launch reserves the LDS of its largest bodies' lanes, so
// one body of hundreds of atoms (16 lanes at most by default) takes the other
// bodies' waves.  Steps in registers and launched, us a step, beside a body of
// 280, 400 and 500 atoms in mixed precision (4, 3 and 2 waves per CU): 1M waters
// under NO-SQUISH(10) 46, 59 and 85, launched 59 to 60; exact rotation 44, 54
// and 73, launched 70; 300k waters 16, 20 and 28, launched 25 to 26; 100k waters
// 7, 9 and 11.5, launched 18 to 21; 200k mixed bodies (4063 tiles) 16, 19 and 27,
// launched 33.  So at 2 waves at most 8 turns.  In double precision, where a
// launched step moves twice the bytes, the registers win at 2 waves too (1M
// waters and 280 atoms 104 and 92, launched 136 and 131).
bool steps_lds_pays(int precision, size_t lds, int bodyTiles) {
    const int waves = waves_by_lds(lds);
    return precision != 0 || waves >= 3 || bodyTiles <= 8 * 256 * waves;
}

// (boundaries, flags) of the launches that carry a system through
// `boundaries` step boundaries, the last one's with STEPS_LAST
template <class Launch> static hipError_t steps_launches(int boundaries, Launch&& launch) {
    int flags = STEPS_FIRST;
    do {
        const int n = boundaries < kStepsPerLaunch ? boundaries : kStepsPerLaunch;
        boundaries -= n;
        if (boundaries == 0) flags |= STEPS_LAST;
        launch(n, flags);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        flags = 0;
    } while (boundaries > 0);
    return hipSuccess;
}

hipError_t launch_steps(int precision, int rotationMode, const DevSys* systems, const Tile* tiles, int numTiles,
                        int boundaries, int atomsPerLane, int sitesPerLane, hipStream_t stream, int adopted) {
    if (numTiles <= 0) return hipSuccess;
    const size_t lds = steps_lds_bytes(precision, atomsPerLane, sitesPerLane);
    if (lds > kStepsLdsMax || (adopted && sitesPerLane)) return hipErrorInvalidValue;
    return steps_launches(boundaries, [&](int n, int flags) {
        if (adopted)
            steps_for<AdoptedAtoms, false>(precision, rotationMode, numTiles, lds, stream, systems, tiles, numTiles, n, flags);
        else if (sitesPerLane)
            steps_for<SoaAtoms, true>(precision, rotationMode, numTiles, lds, stream, systems, tiles, numTiles, n, flags);
        else
            steps_for<SoaAtoms, false>(precision, rotationMode, numTiles, lds, stream, systems, tiles, numTiles, n, flags);
    });
}

template <class Real>
static void cluster_steps_classes(const DevSys* systems, const Tile* tiles, const int* counts, int boundaries,
                                  int flags, hipStream_t stream) {
    auto go = [&](auto kernel, int n) {
        if (n) kernel<<<n, kStepsBlock, 0, stream>>>(systems, tiles, boundaries, flags);
        tiles += n;
    };
    go(k_cluster_steps<Real, 2>, counts[0]);
    go(k_cluster_steps<Real, 3>, counts[1]);
    go(k_cluster_steps<Real, 4>, counts[2]);
}

// One launch for both takes as long as the longer, where two take the sum
// (10k four-site waters and 2000 triangles, 49 boundaries: 203 + 342 us, 345
// together).  Its registers allow 2 waves per SIMD, where the bodies alone run
// 4, and every workgroup has the bodies' LDS: so while all of its workgroups
// are resident at once on 256 CUs.  Clusters of 4 atoms need more registers
// than that.
static bool steps_together(int numTiles, const int* counts, size_t lds) {
    const int waves = waves_by_lds(lds);
    return counts[2] == 0 && numTiles + counts[0] + counts[1] <= 256 * (waves < 8 ? waves : 8);
}

hipError_t launch_steps_with_clusters(int precision, int rotationMode, const DevSys* systems, const Tile* tiles,
                                      int numTiles, const Tile* clusterTiles, const int* counts, int boundaries,
                                      int atomsPerLane, int sitesPerLane, hipStream_t stream) {
    const size_t lds = steps_lds_bytes(precision, atomsPerLane, sitesPerLane);
    if (lds > kStepsLdsMax || counts[3]) return hipErrorInvalidValue;
    if (steps_together(numTiles, counts, lds)) {
        const int nc = counts[0] + counts[1];
        return steps_launches(boundaries, [&](int n, int flags) {
            auto go = [&](auto kernel) {
                step_kernel_lds(kernel, nc + numTiles, kStepsBlock, lds, stream, systems, tiles, clusterTiles, nc, n,
                                flags);
            };
            if (precision == 0) {
                if (rotationMode == 0) go(k_steps_mixed<float, true>);
                else go(k_steps_mixed<float, false>);
            } else {
                if (rotationMode == 0) go(k_steps_mixed<double, true>);
                else go(k_steps_mixed<double, false>);
            }
        });
    }
    hipError_t e = launch_steps(precision, rotationMode, systems, tiles, numTiles, boundaries, atomsPerLane,
                                sitesPerLane, stream, 0);
    if (e != hipSuccess) return e;
    return steps_launches(boundaries, [&](int n, int flags) {
        if (precision == 0) cluster_steps_classes<float>(systems, clusterTiles, counts, n, flags, stream);
        else cluster_steps_classes<double>(systems, clusterTiles, counts, n, flags, stream);
    });
}

hipError_t launch_reduce(const DevSys* systems, const int* nslots, int numSystems, int which, double* out,
                         hipStream_t stream) {
    if (numSystems <= 0) return hipSuccess;
    k_reduce<<<numSystems, 256, 0, stream>>>(systems, nslots, 0, which, out);
    return hipGetLastError();
}

hipError_t launch_reduce_one(const DevSys* sys, int nslots, int which, double* out, hipStream_t stream) {
    k_reduce<<<1, 256, 0, stream>>>(sys, nullptr, nslots, which, out);
    return hipGetLastError();
}

hipError_t launch_copy(const void* src, void* dst, size_t bytes, hipStream_t stream) {
    size_t n = bytes / sizeof(float4);
    int grid = (int)((n + 255) / 256 < 8192 ? (n + 255) / 256 : 8192);
    if (grid < 1) grid = 1;
    k_copy<<<grid, 256, 0, stream>>>(reinterpret_cast<const float4*>(src), reinterpret_cast<float4*>(dst), n);
    return hipGetLastError();
}

}  // namespace rbhip
