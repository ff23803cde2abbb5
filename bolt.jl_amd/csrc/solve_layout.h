#ifndef BOLT_SOLVE_LAYOUT_H
#define BOLT_SOLVE_LAYOUT_H

#include "solver_common.h"

// The FP64 integrator's LDS layout and kernel lookup; the kernel is in solve.hip.

// LDS workspace: 30 vectors of NS doubles (NS even: 16-byte loads; rows n..NS-1
// stay zero, so a lane whose rows reach past n reads the identity), then the
// momentum-bin arrays, laid out for NQ bins.  NS and NQ are compile-time: every
// access is then a row's or bin's address plus an immediate offset, where
// runtime strides had the compiler keep an address register per vector and row
// (85 spilled registers at n = 323).
template <int NS, int NQ>
struct WSN {
    static constexpr int kt = (K_Q0 + 2 * NQ + 1) & ~1;  // doubles per scalar table
    static constexpr int ns = NS, NV = 30;
    static constexpr int T0 = NV * NS, XC0 = T0 + 10 * CB, RED0 = XC0 + 5 * NXC, K0 = RED0 + 24, Q0 = K0 + 6 * kt,
                         E0 = Q0 + 27 * NQ, I0 = E0 + NWAVE * (kt + 4 * NQ);
    double* b;
    int n, nq;
    __host__ __device__ double* vec(int i) const { return b + i * NS; }
    __host__ __device__ double* u(int p) const { return vec(p); }      // state, two buffers
    __host__ __device__ double* f(int p) const { return vec(2 + p); }  // derivative, two buffers
    __host__ __device__ double* arg() const { return vec(4); }         // stage argument; the embedded error
    __host__ __device__ double* w() const { return vec(5); }           // stage right-hand side and solution
    __host__ __device__ double* c(int r) const { return vec(6 + r); }  // border columns' solutions
    __host__ __device__ double* cS() const { return c(0); }
    __host__ __device__ double* cP() const { return c(1); }
    __host__ __device__ double* cPi() const { return c(2); }
    __host__ __device__ double* rcp_(int j) const { return vec(9 + j); }
    __host__ __device__ double* tail() const { return b + T0; }
    template <class T> __host__ __device__ BandsT<T> bandsT(int s) const {
        BandsT<T> B;
        B.l1 = vec(15 + 3 * s); B.d = B.l1 + NS; B.u1 = B.d + NS;
        B.l2c = tail() + 2 * CB * s; B.u2c = B.l2c + CB;
        return B;
    }
    __host__ __device__ double* xcs(int s) const { return b + XC0 + NXC * s; }
    __host__ __device__ double* red() const { return b + RED0; }     // [24]: 0..11 border, 16..19 norm
    __host__ __device__ double* dump() const { return red() + 15; }  // a slot nobody reads
    __host__ __device__ double* ktab(int s) const { return b + K0 + kt * s; }
    __host__ __device__ double* kcur() const { return ktab(5); }
    __host__ __device__ double* q() const { return b + Q0; }
    __host__ __device__ double* df0() const { return b + Q0 + NQ; }
    __host__ __device__ double* base() const { return b + Q0 + 2 * NQ; }
    __host__ __device__ double* qe() const { return b + Q0 + 3 * NQ; }
    __host__ __device__ double* qst_base(int s) const { return b + Q0 + (7 + 4 * s) * NQ; }
    // a q-set's four arrays are nq apart (qfill_one)
    __host__ __device__ static QSet qset(const double* p, int nq) {
        QSet Q; Q.qe = p; Q.eqdf = p + nq; Q.sw = p + 2 * nq; Q.rw = p + 3 * nq;
        return Q;
    }
    __host__ __device__ QSet qcur() const { return qset(qe(), nq); }
    __host__ __device__ QSet qst(int s) const { return qset(qst_base(s), nq); }
    // dense output, per wavefront: a scalar table and a q-set
    __host__ __device__ double* esc(int wv) const { return b + E0 + (kt + 4 * NQ) * wv; }
    __host__ __device__ int* kinds() const { return (int*)(b + I0); }
    __host__ __device__ int* seg() const { return kinds() + NS; }
    __host__ __device__ int* misc() const { return seg() + 2 * MAXSEG; }
    __host__ __device__ int* desc() const { return (int*)w(); }  // read by setup_rows alone
    __host__ __device__ unsigned short* place() const { return (unsigned short*)(misc() + 4); }  // row -> Bolt's index
    static constexpr size_t bytes = sizeof(double) * I0 + sizeof(int) * (NS + 2 * MAXSEG + 4) + 2 * NS;
    static constexpr int nmax = NS - SR_MAX;  // longest state
};
// The layouts: up to 256 rows (one owned row per thread; Bolt's default ℓᵧ = 8 is
// n = 197), up to 368 (ℓᵧ = ℓ_ν = 50, ℓ_mν = 10 is 323), up to 512 (plin's defaults
// are 473), and any hierarchy LDS can hold.  The strides spread the LU lanes'
// rows (stage points 3·NS apart) over the banks.
using WSN0 = WSN<278, 16>;
using WSN1 = WSN<376, 16>;
using WSN2 = WSN<524, 16>;
using WSN3 = WSN<538, 48>;
#define WSN_LAYOUTS 4
__host__ __device__ inline int wsn_layout(int n, int nq) {
    return nq > 16 ? 3 : n <= NTHR ? 0 : n <= WSN1::nmax ? 1 : n <= 2 * NTHR ? 2 : 3;
}
__host__ __device__ inline size_t wsn_bytes(int layout) {
    return layout == 0 ? WSN0::bytes : layout == 1 ? WSN1::bytes : layout == 2 ? WSN2::bytes : WSN3::bytes;
}

// the kernel with SR = 6, 7 or 8 scan rows per lane for a layout (solve.hip)
const void* solver_kernel_sr6(int layout);
const void* solver_kernel_sr7(int layout);
const void* solver_kernel_sr8(int layout);
inline const void* solver_kernel(int sr, int layout) {
    return sr == 8 ? solver_kernel_sr8(layout) : sr == 7 ? solver_kernel_sr7(layout) : solver_kernel_sr6(layout);
}

// the tangent-linear solve's kernel, or the FP32 solve mode's (boltsolve.hip)
const void* boltsolve_kernel(bool tan);

#endif  // BOLT_SOLVE_LAYOUT_H
