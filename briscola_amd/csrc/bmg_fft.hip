// FFT Poisson solver on one MI355X: the reference's FFTPoissonSolver
// (src/briscolaFiniteVolume/solvers/PoissonSolvers/FFTPoissonSolver/) for a
// rectilinear mesh with at least two uniform directions, solving
// div(grad x) = -b in its finite-difference form.
//
// Steps (one stream, no host synchronisation inside a solve):
//   1. right-hand side -b minus the boundary terms of the boundary cells
//      (FFTPoissonSolver.C:123-180), two neighbouring planes of the
//      tridiagonal axis s as the real and imaginary part of one complex
//      plane E[s/2][a][c] (a and c the transformed axes).  Every transform
//      is real-linear, so the pair costs one complex FFT:
//        periodic axis: DFT;
//        Neumann or Dirichlet pair: DCT-II (FFTW REDFT10) of the values, or
//          DST-II (RODFT10) as the DCT-II of the values with alternating
//          signs and the modes reversed, from the N-point FFT of the values
//          reordered even ascending, odd descending (Makhoul 1980);
//        Neumann-Dirichlet: DCT-IV (REDFT11) from the 2N-point FFT of the
//          values times e^{-i pi n/2N}, zero-padded; Dirichlet-Neumann:
//          DST-IV (RODFT11), the DCT-IV of the reversed values with
//          alternating signs of the modes;
//   2. one batched 2-D complex FFT over (a, c) (rocFFT);
//   3. the modes from the spectrum (a mode and its mirror images share one
//      thread, so every element is read once): two real numbers per complex
//      one, X[s][k1][k2] real -- a conjugate pair of periodic modes is held
//      as its real and its imaginary part;
//   4. per real mode the tridiagonal solve along s with the reference's
//      coefficients, boundary rows, pinned zero mode and, for a periodic s,
//      its cyclic two-solve variant (tridiagonalSolver.C:14-475);
//   5. the spectrum from the modes and one batched inverse 2-D FFT;
//   6. its real and imaginary parts into the two planes of x, then every
//      ghost of x refreshed (x.correctBoundaryConditions(),
//      FFTPoissonSolver.C:437-440).
// Every boundary pair is taken on every axis.
//
// All steps are bound by memory: 8 bytes per cell and array.  Against a
// complex array per plane, extended to 2N or 4N along Neumann and Dirichlet
// axes and solved as complex lines, the 256^3 channel went from 1660 us to
// 592 us and a 125x90x154 box with cosine, quarter-wave and sine axes from
// 590 us to 154 us.
#include "bmg_context.h"

#include <rocfft/rocfft.h>

#include <cmath>
#include <mutex>

namespace bmg {

namespace {

// Axis codes of FourierTransforms.C:133-215.
enum { C_DD = 1, C_NN = 2, C_DN = 3, C_ND = 4, C_PER = 5 };

int axisCode(int lo, int hi)
{
    if (lo == PER) return C_PER;
    if (lo == DIR) return hi == DIR ? C_DD : C_DN;
    return hi == DIR ? C_ND : C_NN;
}

struct C2 {
    double x, y;
};

__device__ __forceinline__ C2 cmul(C2 a, C2 b)
{
    return C2{a.x*b.x - a.y*b.y, a.x*b.y + a.y*b.x};
}

// a times the conjugate of b
__device__ __forceinline__ C2 cmulc(C2 a, C2 b)
{
    return C2{a.x*b.x + a.y*b.y, a.y*b.x - a.x*b.y};
}

__device__ __forceinline__ C2 cadd(C2 a, C2 b)
{
    return C2{a.x + b.x, a.y + b.y};
}

__device__ __forceinline__ C2 csub(C2 a, C2 b)
{
    return C2{a.x - b.x, a.y - b.y};
}

__device__ __forceinline__ C2 chalf(C2 a) { return C2{0.5*a.x, 0.5*a.y}; }

// i a
__device__ __forceinline__ C2 cmuli(C2 a) { return C2{-a.y, a.x}; }

// A transformed axis: n values, FFT length L, and its tables (device):
// tw[j] = e^{-i pi j/2n} (Neumann and Dirichlet pairs, j <= n/2),
// e^{-i pi (2j+1)/4n} (quarter wave, j < n); pad[j] = e^{-i pi j/2n} (quarter
// wave, j < n); lam[k] the eigenvalue of mode k over the squared width.
struct FftAxis {
    int n, L, code;
    const C2* tw;
    const C2* pad;
    const double* lam;
};

struct FftGeom {
    int N[3], P[3];
    int s, d1, d2;          // tridiagonal axis, transformed axes
    int ns, np;             // planes, plane pairs
    FftAxis a1, a2;         // along d1 and d2
    int codes;
    int bc[6];
    double bcval[6];
    double hwall[6];        // width of the boundary cell of each face
    double dT;              // deltaT*dtFrac of the time term; 0: none
    int oy, oz;             // y and z of a launch's first workgroup
};

__host__ __device__ inline bool halfWave(int code)
{
    return code == C_NN || code == C_DD;
}

__host__ __device__ inline bool quarterWave(int code)
{
    return code == C_ND || code == C_DN;
}

// Position of value a in the FFT's input and its factor.
__device__ __forceinline__ int inputPos(const FftAxis& t, int a, C2& w)
{
    w = C2{1.0, 0.0};
    if (t.code == C_PER) return a;
    if (halfWave(t.code))
    {
        if (t.code == C_DD && (a & 1)) w.x = -1.0;
        return a & 1 ? t.n - 1 - (a >> 1) : a >> 1;
    }
    const int q = t.code == C_DN ? t.n - 1 - a : a;
    w = t.pad[q];
    return q;
}

// Cell (i, j, k) of plane q along axis S, position (a, c) on the others.
template <int S>
__device__ __forceinline__ void cellOf(int q, int a, int c, int g[3])
{
    g[0] = S == 0 ? q : a;
    g[1] = S == 0 ? a : (S == 1 ? q : c);
    g[2] = S == 2 ? q : c;
}

// The thread's (a, c, pair): lanes along c, or with S = 2 (c is then not
// the contiguous axis) 16 of c by 4 pairs, so that reads along the
// contiguous s and writes along c both fill 64-byte lines.
template <int S>
__device__ __forceinline__ void cellThread(const FftGeom& G, int& a, int& c,
                                           int& p)
{
    a = G.oy + blockIdx.y;
    if (S == 2)
    {
        c = blockIdx.x*16 + (threadIdx.x & 15);
        p = (G.oz + blockIdx.z)*16 + (threadIdx.x >> 4);
    }
    else
    {
        c = blockIdx.x*256 + threadIdx.x;
        p = G.oz + blockIdx.z;
    }
}

// Right-hand side of the interior cell g (0-based).
__device__ __forceinline__ double rhsValue(const FftGeom& G, const int g[3],
                                           const double* b, const double* x,
                                           const double* xold)
{
    const long sI = (long)G.P[1]*G.P[2], sJ = G.P[2];
    const long st[3] = {sI, sJ, 1};
    const long c = (g[0] + 1)*sI + (g[1] + 1)*sJ + (g[2] + 1);
    double f = b ? -b[c] : 0.0;
    // ddt: minus x.oldTime()/(deltaT*dtFrac) (FFTPoissonSolver.C:116-131)
    if (xold) f = f - xold[c]/G.dT;
#pragma unroll
    for (int face = 0; face < 6; face++)
    {
        const int d = face >> 1, side = face & 1;
        if (G.bc[face] == PER || g[d] != (side ? G.N[d] - 1 : 0)) continue;
        const double h = G.hwall[face];
        const double sq = h*h;
        const double xg = x[c + (side ? st[d] : -st[d])];
        const double xc = x[c];
        const double term = G.bc[face] == DIR ? (xg + xc)/sq : (xg - xc)/sq;
        f -= term;
    }
    return f;
}

// Step 1; the second half of a quarter-wave axis (zero) included.
template <int S>
__global__ __launch_bounds__(256) void k_fft_rhs(FftGeom G, const double* b,
                                                 const double* x,
                                                 const double* xold, C2* E)
{
    int a, c, p;
    cellThread<S>(G, a, c, p);
    if (c >= G.a2.L || p >= G.np) return;
    C2* Ep = E + (size_t)p*G.a1.L*G.a2.L;
    if (a >= G.a1.n || c >= G.a2.n)
    {
        // only quarter-wave axes have L > n; their padding keeps its place
        // whatever the other axis' reordering
        Ep[(size_t)a*G.a2.L + c] = C2{0.0, 0.0};
        return;
    }
    int g[3];
    cellOf<S>(2*p, a, c, g);
    const double f0 = rhsValue(G, g, b, x, xold);
    double f1 = 0.0;
    if (2*p + 1 < G.ns)
    {
        cellOf<S>(2*p + 1, a, c, g);
        f1 = rhsValue(G, g, b, x, xold);
    }
    C2 w1, w2;
    const int p1 = inputPos(G.a1, a, w1), p2 = inputPos(G.a2, c, w2);
    Ep[(size_t)p1*G.a2.L + p2] = cmul(cmul(w1, w2), C2{f0, f1});
}

// The elements a thread of steps 3 and 5 owns along one axis: index j and
// its mirror image m (-1: none, as index 0 and the middle of an even length
// have), and the modes they give: j itself and, for
// a Neumann or Dirichlet pair or a periodic axis, the image.
struct Orbit {
    int j, m;
};

__host__ __device__ inline int orbits(const FftAxis& t)
{
    return quarterWave(t.code) ? t.n : t.n/2 + 1;
}

__device__ __forceinline__ Orbit orbit(const FftAxis& t, int j)
{
    if (quarterWave(t.code)) return Orbit{j, 2*t.n - 1 - j};
    const int m = t.n - j;
    return Orbit{j, j == 0 || m == j ? -1 : m};
}

// Output index of transform index m (a Dirichlet pair's DST-II modes are
// the DCT-II's in reverse).
__device__ __forceinline__ int modeIndex(const FftAxis& t, int m)
{
    return t.code == C_DD ? t.n - 1 - m : m;
}

// Transform values of an orbit from its spectrum elements u (index j) and v
// (index m), in place: (X_j, X_m).  j == m: u alone.
__device__ __forceinline__ void fromSpectrum(const FftAxis& t, const Orbit& o,
                                             C2& u, C2& v)
{
    if (t.code == C_PER) return;
    if (quarterWave(t.code))
    {
        const C2 w = t.tw[o.j];
        u = chalf(cadd(cmul(w, u), cmulc(v, w)));
        if (t.code == C_DN && (o.j & 1)) u = C2{-u.x, -u.y};
        return;
    }
    const C2 w = t.tw[o.j];
    if (o.m < 0) v = u;
    const C2 a = cmul(w, u), b = cmulc(v, w);
    u = chalf(cadd(a, b));
    v = cmuli(chalf(csub(a, b)));
}

// Spectrum elements (index j, index m) of the inverse FFT's input from the
// transform values; quarter wave: u at j, nothing at the image (the padding).
__device__ __forceinline__ void toSpectrum(const FftAxis& t, const Orbit& o,
                                           C2& u, C2& v)
{
    if (t.code == C_PER) return;
    if (quarterWave(t.code))
    {
        if (t.code == C_DN && (o.j & 1)) u = C2{-u.x, -u.y};
        u = cmulc(u, t.pad[o.j]);
        v = C2{0.0, 0.0};
        return;
    }
    if (o.j == 0) return;
    const C2 w = t.tw[o.j];
    if (o.m < 0) v = u;
    const C2 iv = cmuli(v);
    const C2 a = csub(u, iv), b = cadd(u, iv);
    u = cmulc(a, w);
    v = cmul(b, w);
}

// Where the two planes' values of a transform value go in X: with a periodic
// axis the value at (k1, k2) and at its conjugate partner (the periodic
// indices negated) are Z = A + iB and Z' = conj A + i conj B of the planes'
// modes A and B, held as Re at one and Im at the other.
__device__ __forceinline__ void storeModes(const FftGeom& G, double* X, int p,
                                           int i1, int i2, double v0, double v1)
{
    const size_t nm = (size_t)G.a1.n*G.a2.n;
    const size_t at = (size_t)(2*p)*nm + (size_t)i1*G.a2.n + i2;
    X[at] = v0;
    if (2*p + 1 < G.ns) X[at + nm] = v1;
}

__device__ __forceinline__ C2 loadModes(const FftGeom& G, const double* X,
                                        int p, int i1, int i2)
{
    const size_t nm = (size_t)G.a1.n*G.a2.n;
    const size_t at = (size_t)(2*p)*nm + (size_t)i1*G.a2.n + i2;
    return C2{X[at], 2*p + 1 < G.ns ? X[at + nm] : 0.0};
}

// The orbits a thread owns: along axis 1 and 2 the pairs (j, image), and the
// four combinations (j1,j2), (m1,j2), (j1,m2), (m1,m2), here e0 to e3 (held
// one by one: an array ends up in scratch memory).
struct OrbitPair {
    Orbit o1, o2;
    bool m1, m2;     // the images exist
};

__device__ __forceinline__ bool orbitThread(const FftGeom& G, OrbitPair& q,
                                            int& p)
{
    const int n2 = orbits(G.a2);
    const unsigned t = blockIdx.x*256 + threadIdx.x;
    const int j1 = int(t/unsigned(n2)), j2 = int(t - unsigned(j1)*n2);
    p = G.oy + blockIdx.y;
    if (j1 >= orbits(G.a1)) return false;
    q.o1 = orbit(G.a1, j1);
    q.o2 = orbit(G.a2, j2);
    q.m1 = q.o1.m >= 0;
    q.m2 = q.o2.m >= 0;
    return true;
}

// A complex value and its conjugate partner -> the planes' modes, two real
// numbers each (self: the value is its own partner).
__device__ __forceinline__ void splitPlanes(const FftGeom& G, double* X, int p,
                                            C2 z, int i1, int i2, C2 zp,
                                            int k1, int k2, bool self)
{
    if (self)
    {
        storeModes(G, X, p, i1, i2, z.x, z.y);
        return;
    }
    // A = (Z + conj Z')/2, B = (Z - conj Z')/2i
    storeModes(G, X, p, i1, i2, 0.5*(z.x + zp.x), 0.5*(z.y + zp.y));
    storeModes(G, X, p, k1, k2, 0.5*(z.y - zp.y), 0.5*(zp.x - z.x));
}

// The inverse: Z and its partner Z' from the two real numbers r and m at
// their indices, Z = A + iB, Z' = conj A + i conj B, A = r.x + i m.x,
// B = r.y + i m.y (self: Z alone, both real).
__device__ __forceinline__ C2 joinFirst(C2 r, C2 m, bool self)
{
    return C2{self ? r.x : r.x - m.y, self ? r.y : m.x + r.y};
}

__device__ __forceinline__ C2 joinSecond(C2 r, C2 m)
{
    return C2{r.x + m.y, r.y - m.x};
}

// Step 3.
__global__ __launch_bounds__(256) void k_fft_modes(FftGeom G, const C2* E,
                                                   double* X)
{
    OrbitPair q;
    int p;
    if (!orbitThread(G, q, p)) return;
    const C2* Ep = E + (size_t)p*G.a1.L*G.a2.L;
    // an index without an image repeats its element
    const size_t r1 = (size_t)q.o1.j*G.a2.L;
    const size_t r1m = (size_t)(q.m1 ? q.o1.m : q.o1.j)*G.a2.L;
    const int c2 = q.o2.j, c2m = q.m2 ? q.o2.m : q.o2.j;
    C2 e0 = Ep[r1 + c2], e1 = Ep[r1m + c2], e2 = Ep[r1 + c2m],
       e3 = Ep[r1m + c2m];
    fromSpectrum(G.a1, q.o1, e0, e1);
    fromSpectrum(G.a1, q.o1, e2, e3);
    fromSpectrum(G.a2, q.o2, e0, e2);
    fromSpectrum(G.a2, q.o2, e1, e3);
    const bool per1 = G.a1.code == C_PER, per2 = G.a2.code == C_PER;
    const bool q1 = quarterWave(G.a1.code), q2 = quarterWave(G.a2.code);
    // modes along each axis: j always; the image where there is one, but a
    // quarter wave's
    const bool h1 = q.m1 && !q1, h2 = q.m2 && !q2;
    const int i1 = modeIndex(G.a1, q.o1.j), i2 = modeIndex(G.a2, q.o2.j);
    const int k1 = h1 ? modeIndex(G.a1, q.o1.m) : i1;
    const int k2 = h2 ? modeIndex(G.a2, q.o2.m) : i2;
    if (per1 && per2)
    {
        splitPlanes(G, X, p, e0, i1, i2, h1 ? (h2 ? e3 : e1) : e2, k1,
                    k2, !h1 && !h2);
        if (h1 && h2) splitPlanes(G, X, p, e1, k1, i2, e2, i1, k2, false);
    }
    else if (per1)
    {
        splitPlanes(G, X, p, e0, i1, i2, e1, k1, i2, !h1);
        if (h2) splitPlanes(G, X, p, e2, i1, k2, e3, k1, k2, !h1);
    }
    else if (per2)
    {
        splitPlanes(G, X, p, e0, i1, i2, e2, i1, k2, !h2);
        if (h1) splitPlanes(G, X, p, e1, k1, i2, e3, k1, k2, !h2);
    }
    else
    {
        storeModes(G, X, p, i1, i2, e0.x, e0.y);
        if (h1) storeModes(G, X, p, k1, i2, e1.x, e1.y);
        if (h2) storeModes(G, X, p, i1, k2, e2.x, e2.y);
        if (h1 && h2) storeModes(G, X, p, k1, k2, e3.x, e3.y);
    }
}

// Step 5; the whole extended spectrum is written.
__global__ __launch_bounds__(256) void k_fft_spectrum(FftGeom G,
                                                      const double* X, C2* E)
{
    OrbitPair q;
    int p;
    if (!orbitThread(G, q, p)) return;
    C2* Ep = E + (size_t)p*G.a1.L*G.a2.L;
    const bool per1 = G.a1.code == C_PER, per2 = G.a2.code == C_PER;
    const bool q1 = quarterWave(G.a1.code), q2 = quarterWave(G.a2.code);
    const bool h1 = q.m1 && !q1, h2 = q.m2 && !q2;
    const int i1 = modeIndex(G.a1, q.o1.j), i2 = modeIndex(G.a2, q.o2.j);
    const int k1 = h1 ? modeIndex(G.a1, q.o1.m) : i1;
    const int k2 = h2 ? modeIndex(G.a2, q.o2.m) : i2;
    // all four modes loaded before any branch (an index without an image
    // repeats)
    const C2 ii = loadModes(G, X, p, i1, i2), ki = loadModes(G, X, p, k1, i2);
    const C2 ik = loadModes(G, X, p, i1, k2), kk = loadModes(G, X, p, k1, k2);
    // no periodic axis: the values themselves
    C2 e0 = ii, e1 = ki, e2 = ik, e3 = kk;
    if (per1 && per2)
    {
        // partners (j1,j2)-(m1,m2) and (m1,j2)-(j1,m2); with one image
        // missing the first alone, at whichever index has one
        const C2 zp = joinSecond(ii, kk);
        const bool both = h1 && h2;
        e0 = joinFirst(ii, kk, !h1 && !h2);
        e1 = both ? joinFirst(ki, ik, false) : zp;
        e2 = both ? joinSecond(ki, ik) : zp;
        e3 = zp;
    }
    else if (per1)
    {
        e0 = joinFirst(ii, ki, !h1);
        e1 = joinSecond(ii, ki);
        e2 = joinFirst(ik, kk, !h1);
        e3 = joinSecond(ik, kk);
    }
    else if (per2)
    {
        e0 = joinFirst(ii, ik, !h2);
        e2 = joinSecond(ii, ik);
        e1 = joinFirst(ki, kk, !h2);
        e3 = joinSecond(ki, kk);
    }
    toSpectrum(G.a1, q.o1, e0, e1);
    toSpectrum(G.a1, q.o1, e2, e3);
    toSpectrum(G.a2, q.o2, e0, e2);
    toSpectrum(G.a2, q.o2, e1, e3);
    const size_t r1 = (size_t)q.o1.j*G.a2.L;
    const size_t r1m = (size_t)(q.m1 ? q.o1.m : 0)*G.a2.L;
    Ep[r1 + q.o2.j] = e0;
    if (q.m1) Ep[r1m + q.o2.j] = e1;
    if (q.m2) Ep[r1 + q.o2.m] = e2;
    if (q.m1 && q.m2) Ep[r1m + q.o2.m] = e3;
}

// A row of the tridiagonal systems along s: couplings to the rows above and
// below, and what its diagonal takes off the modes' eigenvalue (the boundary
// rows as tridiagonalSolver.C:107-250).
struct FftRow {
    double up, down, east, west;
};

// Step 4: one thread per real mode, lanes along k2.  X: the transformed
// right-hand side in, the solution out; R: reciprocals of the eliminated
// diagonal; V: the cyclic auxiliary solution.  One division per row serves
// its elimination and its back substitution.  Few wavefronts are in flight
// (one per 64 modes), so each loads the next eight rows while it eliminates
// eight: 256^3 256 us without that, 164 us with it (six arrays of 134 MB).
template <bool CYC>
__global__ __launch_bounds__(64) void k_fft_tridiag(
    FftGeom G, double* __restrict__ X, double* __restrict__ R,
    double* __restrict__ V, const FftRow* __restrict__ row, double pin)
{
    const int k2 = blockIdx.x*64 + threadIdx.x;
    const int k1 = G.oy + blockIdx.y;
    if (k2 >= G.a2.n) return;
    const size_t nm = (size_t)G.a1.n*G.a2.n;
    const size_t t = (size_t)k1*G.a2.n + k2;
    const double l1 = G.a1.lam[k1], l2 = G.a2.lam[k2];
    const double Lm = l1 + l2;
    // zero mode of a singular system: the first row pinned
    const bool pinned = l1 == 0.0 && l2 == 0.0 &&
                        (G.codes == C_NN || G.codes == C_PER);
    const int ns = G.ns, last = ns - 1;
    // ddt: every diagonal minus 1/(deltaT*dtFrac) (:352, :430), the pinned
    // row included
    const double idT = G.dT != 0.0 ? 1.0/G.dT : 0.0;
    auto diag = [&](int k, const FftRow& w) -> double
    {
        const double d = pinned && k == 0 ? pin : Lm - w.east - w.west;
        return d - idT;
    };
    constexpr int AH = 8;
    constexpr int start = CYC ? 1 : 0;
    // forward elimination (tridiagonalSolver.C:340-346)
    double f = 0.0, r = 0.0, v = 0.0, up = 0.0;
    double nxt[AH], cur[AH];
    auto ahead = [&](int k0, double (&d)[AH])
    {
#pragma unroll
        for (int u = 0; u < AH; u++)
            d[u] = X[(size_t)min(k0 + u, last)*nm + t];
    };
    ahead(start, nxt);
    for (int k0 = start; k0 < ns; k0 += AH)
    {
#pragma unroll
        for (int u = 0; u < AH; u++) cur[u] = nxt[u];
        if (k0 + AH < ns) ahead(k0 + AH, nxt);
#pragma unroll
        for (int u = 0; u < AH; u++)
        {
            const int k = k0 + u;
            if (k >= ns) break;
            const FftRow w = row[k];
            double d = diag(k, w);
            double fk = cur[u];
            double vk = 0.0;
            if (CYC) vk = k == 1 ? -w.down : (k == last ? -w.up : 0.0);
            if (k > start)
            {
                const double m = w.down*r;
                d = d - m*up;
                fk = fk - m*f;
                if (CYC) vk = vk - m*v;
            }
            r = 1.0/d;
            f = fk;
            v = vk;
            up = w.up;
            if (k < last)
            {
                X[(size_t)k*nm + t] = f;
                R[(size_t)k*nm + t] = r;
                if (CYC) V[(size_t)k*nm + t] = v;
            }
        }
    }
    // back substitution (:348-354)
    f = f*r;
    v = v*r;
    X[(size_t)last*nm + t] = f;
    if (CYC) V[(size_t)last*nm + t] = v;
    const double uN = f, vN = v;
    double fn[AH], rn[AH], vn[AH];
    auto behind = [&](int k0)
    {
#pragma unroll
        for (int u = 0; u < AH; u++)
        {
            const size_t at = (size_t)max(k0 - u, start)*nm + t;
            fn[u] = X[at];
            rn[u] = R[at];
            vn[u] = CYC ? V[at] : 0.0;
        }
    };
    if (ns - 2 >= start) behind(ns - 2);
    for (int k0 = ns - 2; k0 >= start; k0 -= AH)
    {
        double fi[AH], ri[AH], vi[AH];
#pragma unroll
        for (int u = 0; u < AH; u++)
        {
            fi[u] = fn[u];
            ri[u] = rn[u];
            vi[u] = vn[u];
        }
        if (k0 - AH >= start) behind(k0 - AH);
#pragma unroll
        for (int u = 0; u < AH; u++)
        {
            const int k = k0 - u;
            if (k < start) break;
            const double c = row[k].up;
            f = (fi[u] - c*f)*ri[u];
            X[(size_t)k*nm + t] = f;
            if (CYC)
            {
                v = (vi[u] - c*v)*ri[u];
                V[(size_t)k*nm + t] = v;
            }
        }
    }
    if constexpr (CYC)
    {
        // reconstruction (tridiagonalSolver.C:418-450); f, v: row 1
        const FftRow w = row[0];
        const double den = (diag(0, w) + w.down*vN) + w.up*v;
        const double p0 = ((X[t] - w.down*uN) - w.up*f)/den;
        X[t] = p0;
#pragma unroll 8
        for (int k = 1; k < ns; k++)
        {
            const size_t at = (size_t)k*nm + t;
            X[at] = X[at] + p0*V[at];
        }
    }
}

// Value (a, c) of a plane pair from the inverse FFT, unscaled: quarter-wave
// axes sum an element and its image, e^{i phi} D_n + e^{-i phi} D_(2N-1-n).
__device__ __forceinline__ C2 outputLine(const FftAxis& t, const C2* line,
                                         int c)
{
    if (t.code == C_PER) return line[c];
    if (halfWave(t.code))
    {
        const C2 v = line[c & 1 ? t.n - 1 - (c >> 1) : c >> 1];
        return t.code == C_DD && (c & 1) ? C2{-v.x, -v.y} : v;
    }
    const int q = t.code == C_DN ? t.n - 1 - c : c;
    const C2 w = t.tw[q];
    return cadd(cmulc(line[q], w), cmul(line[2*t.n - 1 - q], w));
}

// Step 6: the two planes of x.
template <int S>
__global__ __launch_bounds__(256) void k_fft_out(FftGeom G, const C2* E,
                                                 double* x, double scale)
{
    int a, c, p;
    cellThread<S>(G, a, c, p);
    if (c >= G.a2.n || p >= G.np) return;
    const C2* Ep = E + (size_t)p*G.a1.L*G.a2.L;
    const FftAxis& t = G.a1;
    C2 v;
    if (quarterWave(t.code))
    {
        const int q = t.code == C_DN ? t.n - 1 - a : a;
        const C2 w = t.tw[q];
        v = cadd(cmulc(outputLine(G.a2, Ep + (size_t)q*G.a2.L, c), w),
                 cmul(outputLine(G.a2, Ep + (size_t)(2*t.n - 1 - q)*G.a2.L, c),
                      w));
    }
    else
    {
        int q = a;
        if (halfWave(t.code)) q = a & 1 ? t.n - 1 - (a >> 1) : a >> 1;
        v = outputLine(G.a2, Ep + (size_t)q*G.a2.L, c);
        if (t.code == C_DD && (a & 1)) v = C2{-v.x, -v.y};
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
    {
        if (2*p + h >= G.ns) break;
        int g[3];
        cellOf<S>(2*p + h, a, c, g);
        x[((size_t)(g[0] + 1)*G.P[1] + (g[1] + 1))*G.P[2] + (g[2] + 1)] =
            (h ? v.y : v.x)*scale;
    }
}

// Eigenvalue of mode k (tridiagonalSolver.C:31-98).
double eigen(int code, int n, int k)
{
    const double pi = 3.14159265358979323846;
    double sn;
    if (code == C_DD) sn = std::sin((k + 1)*pi/(2.0*n));
    else if (code == C_NN) sn = std::sin(k*pi/(2.0*n));
    else if (code == C_PER) sn = std::sin(std::min(k, n - k)*pi/n);
    else sn = std::sin((2.0*(k + 1) - 1.0)*pi/(4.0*n));
    return -4.0*(sn*sn);
}

// Every ghost of x (meshLevel::correctBoundaryConditions on level 0): face
// ghosts by their condition -- periodic image, Neumann x_P + g/delta with
// delta = 1/h of the mirrored boundary cell, Dirichlet 2v - x_P -- and edge
// and corner ghosts by periodic image when every face they border is
// periodic, else a copy of the adjacent interior cell.
__global__ __launch_bounds__(256) void k_fft_ghosts(FftGeom g, double* x)
{
    // blockIdx.z: the two faces normal to an axis (whole, the lower axis'
    // edges included); blockIdx.y a row, lanes along its last axis
    const int d = blockIdx.z >> 1, side = blockIdx.z & 1;
    const int a1 = d == 0 ? 1 : 0, a2 = d == 2 ? 1 : 2;
    const int u = blockIdx.x*256 + threadIdx.x;
    const int v1 = g.oy + blockIdx.y;
    if (v1 >= g.P[a1] || u >= g.P[a2]) return;
    const int w = side ? g.P[d] - 1 : 0;
    int q[3];
    q[0] = d == 0 ? w : v1;
    q[1] = d == 0 ? v1 : (d == 1 ? w : u);
    q[2] = d == 2 ? w : u;
    const long t = ((long)q[0]*g.P[1] + q[1])*g.P[2] + q[2];
    int bo[3], nout = 0;
    bool allPer = true;
    for (int d = 0; d < 3; d++)
    {
        bo[d] = q[d] == 0 ? -1 : (q[d] == g.P[d] - 1 ? 1 : 0);
        nout += bo[d] != 0;
        if (bo[d] != 0 && g.bc[2*d + (bo[d] > 0)] != PER) allPer = false;
    }
    if (nout == 0) return;
    int sidx[3];
    for (int d = 0; d < 3; d++)
        sidx[d] = allPer ? q[d] - bo[d]*g.N[d] : q[d] - bo[d];
    const double xi = x[((long)sidx[0]*g.P[1] + sidx[1])*g.P[2] + sidx[2]];
    double v = xi;
    if (nout == 1 && !allPer)
    {
        const int d = bo[0] ? 0 : (bo[1] ? 1 : 2);
        const int f = 2*d + (bo[d] > 0);
        if (g.bc[f] == NEU)
        {
            const double delta = 1.0/g.hwall[f];
            v = xi + g.bcval[f]/delta;
        }
        else
            v = 2.0*g.bcval[f] - xi;
    }
    x[t] = v;
}

void rocfftCheck(rocfft_status s, const char* what)
{
    if (s != rocfft_status_success)
        throw Error(BMG_ERR_HIP, std::string("rocFFT ") + what + " failed (" +
                                     std::to_string(int(s)) + ")");
}

std::once_flag g_rocfftSetup;

}  // namespace

}  // namespace bmg

using namespace bmg;

struct bmg_fft
{
    int device = 0;
    hipStream_t stream = nullptr;
    FftGeom g{};
    C2* E = nullptr;       // plane pairs, np x L1 x L2
    double* X = nullptr;   // modes, ns x n1 x n2
    double* R = nullptr;   // reciprocal eliminated diagonals
    double* V = nullptr;   // cyclic auxiliary solution
    double* tables = nullptr;      // twiddles, eigenvalues and rows
    const FftRow* row = nullptr;   // the rows along s
    double pin = 0.0;              // diagonal of the zero mode's pinned row
    void* work = nullptr;
    rocfft_plan fwd = nullptr, bwd = nullptr;
    rocfft_execution_info info = nullptr;

    ~bmg_fft()
    {
        if (fwd) rocfft_plan_destroy(fwd);
        if (bwd) rocfft_plan_destroy(bwd);
        if (info) rocfft_execution_info_destroy(info);
        for (void* p : {(void*)E, (void*)X, (void*)R, (void*)V,
                        (void*)tables, work})
            if (p) (void)hipFree(p);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace bmg {

void fft_create(bmg_fft** out, const bmg_grid* grid)
{
    if (!out || !grid) throw Error(BMG_ERR_ARG, "null pointer");
    std::unique_ptr<bmg_fft> F(new bmg_fft);
    FftGeom& g = F->g;
    std::vector<double> w[3];
    bool uniform[3];
    for (int d = 0; d < 3; d++)
    {
        g.N[d] = grid->n[d];
        g.P[d] = g.N[d] + 2;
        if (g.N[d] < 1 || !grid->vertices[d])
            throw Error(BMG_ERR_ARG, "bad grid");
        w[d].resize(g.N[d]);
        for (int i = 0; i < g.N[d]; i++)
            w[d][i] = grid->vertices[d][i + 1] - grid->vertices[d][i];
        uniform[d] = true;
        for (int i = 0; i < g.N[d]; i++)
            if (std::fabs(w[d][i] - w[d][0]) > 1e-12*std::fabs(w[d][0]))
                uniform[d] = false;
    }
    for (int f = 0; f < 6; f++)
    {
        g.bc[f] = grid->bc[f];
        g.bcval[f] = grid->bc_value[f];
        g.hwall[f] = (f & 1) ? w[f/2].back() : w[f/2].front();
    }
    for (int f = 0; f < 6; f++)
        if ((g.bc[f] == PER) != (g.bc[f ^ 1] == PER))
            throw Error(BMG_ERR_ARG, "periodic faces come in pairs");
    // planner.C:76-117 (one process)
    int nonUniform = 0;
    g.s = -1;
    for (int d = 0; d < 3; d++)
        if (!uniform[d])
        {
            nonUniform++;
            if (g.s < 0) g.s = d;
        }
    if (nonUniform > 1)
        throw Error(BMG_ERR_ARG, "at least two mesh directions must be "
                                 "uniform for the FFT solver");
    if (g.s < 0) g.s = g.N[0] > 1 ? 0 : 2;
    g.d1 = g.s == 0 ? 1 : 0;
    g.d2 = g.s == 2 ? 1 : 2;
    g.ns = g.N[g.s];
    g.np = (g.ns + 1)/2;
    g.codes = axisCode(g.bc[2*g.s], g.bc[2*g.s + 1]);
    if (g.ns < 2 || (g.codes == C_PER && g.ns < 3))
        throw Error(BMG_ERR_ARG, "too few cells along the tridiagonal axis");
    FftAxis* ax[2] = {&g.a1, &g.a2};
    const int dd[2] = {g.d1, g.d2};
    std::vector<double> tables;
    size_t at[2][3];
    for (int t = 0; t < 2; t++)
    {
        FftAxis& A = *ax[t];
        const int d = dd[t];
        A.n = g.N[d];
        A.code = axisCode(g.bc[2*d], g.bc[2*d + 1]);
        A.L = quarterWave(A.code) ? 2*A.n : A.n;
        const long double pi = 3.14159265358979323846264338327950288L;
        // tables collected for one upload, in doubles
        auto unit = [&](long double th)
        {
            tables.push_back(double(std::cos(th)));
            tables.push_back(double(std::sin(th)));
        };
        at[t][0] = tables.size();
        if (halfWave(A.code))
            for (int j = 0; j <= A.n/2; j++) unit(-pi*j/(2.0L*A.n));
        if (quarterWave(A.code))
            for (int j = 0; j < A.n; j++) unit(-pi*(2*j + 1)/(4.0L*A.n));
        at[t][1] = tables.size();
        if (quarterWave(A.code))
            for (int j = 0; j < A.n; j++) unit(-pi*j/(2.0L*A.n));
        at[t][2] = tables.size();
        const double sq = w[d][0]*w[d][0];
        for (int k = 0; k < A.n; k++)
            tables.push_back(eigen(A.code, A.n, k)/sq);
        if (tables.size() & 1) tables.push_back(0.0);
    }
    // widths along s with the ghost widths (mirrored, or the periodic
    // images) and their means (tridiagonalSolver.C:112-130)
    const std::vector<double>& ws = w[g.s];
    const int ns = g.ns;
    const bool per = g.codes == C_PER;
    std::vector<double> hg(ns + 2), h(ns), de(ns), dw(ns);
    hg[0] = per ? ws[ns - 1] : ws[0];
    hg[ns + 1] = per ? ws[0] : ws[ns - 1];
    for (int k = 0; k < ns; k++) hg[k + 1] = ws[k];
    for (int k = 0; k < ns; k++)
    {
        h[k] = hg[k + 1];
        de[k] = (hg[k + 1] + hg[k + 2])/2.0;
        dw[k] = (hg[k + 1] + hg[k])/2.0;
    }
    HIPCK(hipGetDevice(&F->device));
    HIPCK(hipStreamCreateWithFlags(&F->stream, hipStreamNonBlocking));
    const size_t nE = size_t(g.np)*g.a1.L*g.a2.L;
    const size_t nX = size_t(ns)*g.a1.n*g.a2.n;
    F->E = devAlloc<C2>(nE);
    F->X = devAlloc<double>(nX);
    F->R = devAlloc<double>(nX);
    F->V = devAlloc<double>(per ? nX : 1);
    std::vector<FftRow> rows(ns);
    for (int k = 0; k < ns; k++)
    {
        FftRow& q = rows[k];
        q.up = 1.0/(h[k]*de[k]);
        q.down = 1.0/(h[k]*dw[k]);
        q.east = q.up;
        q.west = q.down;
        if (per) continue;
        if (k == 0)
            q.west = g.codes == C_DD || g.codes == C_DN ? 2.0/(h[0]*dw[0])
                                                        : 0.0;
        if (k == ns - 1)
            q.east = g.codes == C_DD || g.codes == C_ND ? 2.0/(de[k]*h[k])
                                                        : 0.0;
    }
    F->pin = -1.0/(de[0]*h[0]) - 2.0/(h[0]*dw[0]);
    const size_t atRows = tables.size();
    for (const FftRow& q : rows)
        tables.insert(tables.end(), {q.up, q.down, q.east, q.west});
    F->tables = devUpload(tables);
    for (int t = 0; t < 2; t++)
    {
        ax[t]->tw = reinterpret_cast<const C2*>(F->tables + at[t][0]);
        ax[t]->pad = reinterpret_cast<const C2*>(F->tables + at[t][1]);
        ax[t]->lam = F->tables + at[t][2];
    }
    F->row = reinterpret_cast<const FftRow*>(F->tables + atRows);
    std::call_once(g_rocfftSetup, [] { rocfftCheck(rocfft_setup(), "setup"); });
    // an axis of one point needs no FFT (and two leave none)
    size_t lengths[2], dims = 0;
    for (const FftAxis* A : {&g.a2, &g.a1})
        if (A->L > 1) lengths[dims++] = size_t(A->L);
    if (dims == 0)
    {
        *out = F.release();
        return;
    }
    rocfftCheck(rocfft_plan_create(&F->fwd, rocfft_placement_inplace,
                                   rocfft_transform_type_complex_forward,
                                   rocfft_precision_double, dims, lengths,
                                   size_t(g.np), nullptr), "plan");
    rocfftCheck(rocfft_plan_create(&F->bwd, rocfft_placement_inplace,
                                   rocfft_transform_type_complex_inverse,
                                   rocfft_precision_double, dims, lengths,
                                   size_t(g.np), nullptr), "plan");
    size_t w1 = 0, w2 = 0;
    rocfftCheck(rocfft_plan_get_work_buffer_size(F->fwd, &w1), "work size");
    rocfftCheck(rocfft_plan_get_work_buffer_size(F->bwd, &w2), "work size");
    rocfftCheck(rocfft_execution_info_create(&F->info), "execution info");
    rocfftCheck(rocfft_execution_info_set_stream(F->info, F->stream),
                "stream");
    const size_t wb = std::max(w1, w2);
    if (wb)
    {
        HIPCK(hipMalloc(&F->work, wb));
        rocfftCheck(rocfft_execution_info_set_work_buffer(F->info, F->work,
                                                          wb), "work buffer");
    }
    *out = F.release();
}

void fft_destroy(bmg_fft* F) { delete F; }

// FFTPoissonSolver::solve (FFTPoissonSolver.C:97-465) on device arrays in
// the reference layout; b may be null (b = 0).  With dxold the time term:
// the source minus x_old/dT and every diagonal minus 1/dT, dT =
// deltaT*dtFrac (FFTPoissonSolver.C:116-131, tridiagonalSolver.C:334-352).
void fft_solve_device(bmg_fft* F, const double* db, double* dx,
                      const double* dxold, double dT)
{
    if (!F || !dx) throw Error(BMG_ERR_ARG, "null pointer");
    if (dxold && !(std::isfinite(dT) && dT > 0.0))
        throw Error(BMG_ERR_ARG, "time term needs deltaT*dtFrac > 0");
    FftGeom g = F->g;
    g.dT = dxold ? dT : 0.0;
    hipStream_t s = F->stream;
    auto blocks = [](size_t n, int b) { return unsigned((n + b - 1)/b); };
    // launches whose y and z stay within the device's grid limit (65536),
    // which a long axis exceeds
    auto launch = [&](auto kernel, dim3 grid, unsigned threads, auto... args)
    {
        constexpr unsigned most = 65535;
        for (unsigned z = 0; z < grid.z; z += most)
            for (unsigned y = 0; y < grid.y; y += most)
            {
                g.oy = int(y);
                g.oz = int(z);
                hipLaunchKernelGGL(kernel,
                                   dim3(grid.x, std::min(most, grid.y - y),
                                        std::min(most, grid.z - z)),
                                   dim3(threads), 0, s, g, args...);
                HIPCK(hipGetLastError());
            }
    };
    // steps 1 and 6: a thread per plane pair and position
    auto cells = [&](int L1, int L2)
    {
        return g.s == 2 ? dim3(blocks(L2, 16), L1, blocks(g.np, 16))
                        : dim3(blocks(L2, 256), L1, g.np);
    };
    const dim3 gin = cells(g.a1.L, g.a2.L), gout = cells(g.a1.n, g.a2.n);
    launch(g.s == 0 ? k_fft_rhs<0> : g.s == 1 ? k_fft_rhs<1> : k_fft_rhs<2>,
           gin, 256, db, (const double*)dx, dxold, F->E);
    void* buf[1] = {F->E};
    if (F->fwd)
        rocfftCheck(rocfft_execute(F->fwd, buf, nullptr, F->info), "forward");
    const dim3 gorb(blocks(size_t(orbits(g.a1))*orbits(g.a2), 256), g.np);
    launch(k_fft_modes, gorb, 256, (const C2*)F->E, F->X);
    launch(g.codes == C_PER ? k_fft_tridiag<true> : k_fft_tridiag<false>,
           dim3(blocks(g.a2.n, 64), g.a1.n), 64, F->X, F->R, F->V, F->row,
           F->pin);
    launch(k_fft_spectrum, gorb, 256, (const double*)F->X, F->E);
    if (F->bwd)
        rocfftCheck(rocfft_execute(F->bwd, buf, nullptr, F->info), "inverse");
    const double scale = 1.0/(double(g.a1.n)*double(g.a2.n));
    launch(g.s == 0 ? k_fft_out<0> : g.s == 1 ? k_fft_out<1> : k_fft_out<2>,
           gout, 256, (const C2*)F->E, dx, scale);
    launch(k_fft_ghosts, dim3(blocks(std::max(g.P[1], g.P[2]), 256),
                              std::max(g.P[0], g.P[1]), 6), 256, dx);
    HIPCK(hipStreamSynchronize(s));
}

void fft_solve(bmg_fft* F, const double* b, double* x, const double* xold,
               double dT)
{
    if (!F || !x) throw Error(BMG_ERR_ARG, "null pointer");
    const FftGeom& g = F->g;
    const size_t n = size_t(g.P[0])*g.P[1]*g.P[2];
    double* db = nullptr;
    double* dold = nullptr;
    double* dx = devAlloc<double>(n);
    try
    {
        if (b)
        {
            db = devAlloc<double>(n);
            HIPCK(hipMemcpy(db, b, n*sizeof(double), hipMemcpyHostToDevice));
        }
        if (xold)
        {
            dold = devAlloc<double>(n);
            HIPCK(hipMemcpy(dold, xold, n*sizeof(double),
                            hipMemcpyHostToDevice));
        }
        HIPCK(hipMemcpy(dx, x, n*sizeof(double), hipMemcpyHostToDevice));
        fft_solve_device(F, db, dx, dold, dT);
        HIPCK(hipMemcpy(x, dx, n*sizeof(double), hipMemcpyDeviceToHost));
    }
    catch (...)
    {
        devFree(db);
        devFree(dold);
        devFree(dx);
        throw;
    }
    devFree(db);
    devFree(dold);
    devFree(dx);
}

}  // namespace bmg
