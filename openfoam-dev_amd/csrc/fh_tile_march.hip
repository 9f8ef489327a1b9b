// Marching DIC / DILU and Gauss-Seidel sweeps for hex boxes (the global
// preconditioner passes of the FP64 and FP32 Krylov solvers, the FP64
// Gauss-Seidel smoothers).
//
// The recurrences are those of fh_tile_sweep.hip (DICPreconditioner.C:
// 87-123, DILUPreconditioner.C:88-135, GaussSeidelSmoother.C:66-187,
// symGaussSeidelSmoother.C:66-216): cell (i,j,k) waits for its lower
// neighbours (forward) or upper neighbours (backward, the same in reversed
// coordinates), and each row keeps the reference face order (k, j, i), so
// the results are bitwise those of the sequential loops.
//
// What bounds such a pass is first the chain of dependent cells, then what a
// compute unit can load: most of the chain is the lag between the starts of
// the pencils, and where the packed coefficients come from HBM (they do in a
// solve of a box beyond the last-level cache) a pass takes about a quarter
// longer than launched back to back.  A workgroup therefore owns a pencil of 16 x 16 columns and marches along
// k through the whole box without stopping: four wavefronts compute (16
// columns along i by 4 along j each, lane (i, j) at plane k = step - i -
// 2 j), so the chain has nz + 21 steps per wavefront and no tile to drain
// and refill, and only two directions are left in which a value crosses
// from one workgroup to another.
//   - i-1 comes from the lane beside (DPP row shift; lane 0 of a row takes
//     the pencil's halo as the shift's old value), k-1 is the lane's own
//     last result, j-1 was written to LDS two steps earlier, so its read
//     is issued a step ahead and its latency is off the chain.
//   - The coefficients are packed once per coefficient update, multiplied
//     by rD (the products the reference forms) and in the order the lanes
//     use them (step, lane): every load is contiguous, sixteen steps are in
//     flight in registers.  Absent neighbours and steps outside the box
//     hold zeros, so a step has no branch and no select.
//   - Four input wavefronts load the planes ahead into LDS rings of 64
//     steps (in which the results replace the inputs), take the halo values
//     from the pencils upstream and sum w*r over the finished planes; four
//     output wavefronts publish the pencil's boundary values and write
//     finished planes as whole rows.  With loads and stores apart no load
//     waits behind a store's acknowledgement.
//   - A halo value is its own flag: the slot holds a signalling NaN, which
//     no arithmetic produces, until the producer's store arrives; the
//     consumer puts the NaN back after reading, for the next launch.  The
//     slots are in the order of the reading steps, so both sides move whole
//     rows of them and a reader follows 15 (i) or 6 (j) steps behind.
// Pencils are taken by ticket along their diagonals, so every pencil waited
// on is already running; every wait is bounded.
//
// Measured on an MI355X against the 8 x 8 x 16 tiles of fh_tile_wave.hip,
// launched back to back, and in solves (kernel trace without the launches
// past convergence; the 128^3 PBiCGStab's backward passes take no sum), us
// per pass, forward / backward with its sum:
//                      FP64 here   in a solve  tiles       FP32 here   tiles
//     64^3             70 / 76     70 / 78     130 / 136   56 / 62     118 / 128
//     128^3            152 / 163   193 / 188   288 / 302   121 / 131   286 / 307
//     200 x 150 x 133  208 / 222   273 / 285   382 / 394   180 / 191   379 / 401
//     256^3            493 / 520               641 / 652   342 / 375   604 / 640
// (256^3: 978 and 956 MB of traffic counted, 804 and 938 read or written
// once: the skew's padding and the halos.)
// A Gauss-Seidel row also takes the values on its other side, which the
// sweep does not change before the row is reached (forward: old ones) or at
// all (backward: the forward pass's).  Forward their three products are
// formed ahead in the packed order (the row subtracts them one by one after
// the new values' products), backward the source less the lower products
// is formed ahead as one vector, so a step reads streams only.  Against the
// 16 x 16 x 4 tiles (us per sweep, everything included, forward /
// forward and backward, with the residual of a solver iteration):
//                      here          tiles
//     16^3             33 / 53       77 / 145
//     64^3             113 / 190     386 / 758
//     150 x 100 x 60   213 / 405     532 / 1032
//     256 x 256 x 16   393 / 657     611 / 1188
//     200 x 150 x 133  565 / 878     1035 / 1955
//     256^3            1390 / 2035   2435 / 4350
// (in a solve of 150 x 100 x 60 cells the two kernels alone take 188 and 154
// us, back to back 161 and 134).
// A step takes 0.10 (FP32) to 0.16 us (FP64) in a pencil alone, where a
// compute unit moves 60 to 80 GB/s; a pencil starts about 20 (i) or 47 (j)
// steps and one hand-off through memory after the one before.
#include "fh_tile_march.h"
#include "fh_finalize_dev.h"

namespace fh
{

constexpr int MC = 16;            // pencil width along i and j
constexpr int MW = 4;             // computing wavefronts (4 columns along j each)
constexpr int MG = 4;             // steps per block
constexpr int MD = 4;             // coefficient blocks in flight
constexpr int MSKI = 6, MSKJ = 15; // lags within a wavefront: 2 x 3 along j, 15 along i
constexpr int MSKEW = MSKI + MSKJ; // the last lane's
constexpr int MRS = 64;           // steps of the LDS rings
constexpr int MLAG = 12;          // blocks between staging and summing a plane
constexpr unsigned int M_OOB = 0xF8000000u;   // past every buffer: loads give 0, stores nothing
constexpr uint32_t M_GLOBAL_SPINS = 1u << 20, M_LDS_SPINS = 1u << 24;

template<class T> struct MBits;
template<> struct MBits<double>
{
    typedef unsigned long long U;
    typedef double2 V2;
    static constexpr U sent = 0x7ff4deadbeef0001ull;
    typedef unsigned int B2 __attribute__((ext_vector_type(2)));
    static __device__ double val(U u) { return __longlong_as_double((long long)u); }
    static __device__ U bits(double v) { return (U)__double_as_longlong(v); }
    template<int AUX>
    static __device__ U load(__amdgpu_buffer_rsrc_t r, unsigned int vo, unsigned int so)
    {
        const B2 b = __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, AUX);
        return ((U)b.y << 32) | b.x;
    }
    template<int AUX>
    static __device__ void store(__amdgpu_buffer_rsrc_t r, U v, unsigned int vo, unsigned int so)
    {
        __builtin_amdgcn_raw_buffer_store_b64(B2{(unsigned int)v, (unsigned int)(v >> 32)}, r, vo,
                                              so, AUX);
    }
};
template<> struct MBits<float>
{
    typedef unsigned int U;
    typedef float2 V2;
    static constexpr U sent = 0x7fa0beefu;
    static __device__ float val(U u) { return __uint_as_float(u); }
    static __device__ U bits(float v) { return __float_as_uint(v); }
    template<int AUX>
    static __device__ U load(__amdgpu_buffer_rsrc_t r, unsigned int vo, unsigned int so)
    {
        return __builtin_amdgcn_raw_buffer_load_b32(r, vo, so, AUX);
    }
    template<int AUX>
    static __device__ void store(__amdgpu_buffer_rsrc_t r, U v, unsigned int vo, unsigned int so)
    {
        __builtin_amdgcn_raw_buffer_store_b32(v, r, vo, so, AUX);
    }
};

// cache policy of the halo accesses: device scope (sc1)
constexpr int M_COH = 16;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t m_rsrc(const void* p, unsigned int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}

// what a launch computes
enum
{
    MARCH_FWD = 0,         // forward DIC / DILU pass
    MARCH_BWD = 1,         // backward
    MARCH_GS_FWD = 2,      // Gauss-Seidel rows ascending
    MARCH_GS_BWD = 3       // Gauss-Seidel rows descending (symmetric)
};
template<int MODE> struct MarchMode
{
    static constexpr bool bwd = (MODE & 1) != 0, gs = MODE >= MARCH_GS_FWD;
    static constexpr int na = MODE == MARCH_BWD ? 3 : 4;       // packed coefficients per cell
    static constexpr int no = MODE == MARCH_GS_FWD ? 3 : 0;    // and products of old values
    // coefficient blocks in flight (what the registers hold)
    static constexpr int md = MODE == MARCH_GS_FWD ? 2 : MD;
};

template<class T>
struct MarchArgs
{
    int32_t nx, ny, nz, nPI, nPJ, nPB, nB;
    const T* coef;
    const T* old;          // Gauss-Seidel forward: upper coefficients times old values
    const T* x;
    T* w;
    const T* dotR;
    double* partials;
    T* halo;               // i halos [pencil][nz + 16 steps][16], then j halos
    unsigned long long* ticket;
    unsigned long long ticketBase;
    unsigned int* err;
};

template<class T>
struct MarchShared
{
    // per computing wavefront and step (mod 64): the lanes' inputs, which
    // their results replace (a lane's column is its own bank pair at every
    // step); the halos at the step and row (i) or column (j) that reads them
    T ring[MW][MRS][64];
    T haloI[MRS][MC];
    T haloJ[MRS][MC];
    int inReady[MW];      // blocks staged
    int cStep[MW];        // steps computed
    int oStep[MW];        // steps whose planes are written and boundary published
    int pencil, expired, steps;
    double dot[MW];
};

__device__ __forceinline__ int m_ld(const int* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void m_st(int* p, int v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// lane - 1's value within its row of 16; lane 0 of the row keeps old
__device__ __forceinline__ int m_shr(int v, int old)
{
    return __builtin_amdgcn_update_dpp(old, v, 0x111, 0xf, 0xf, false);
}
__device__ __forceinline__ float m_shr(float v, float old)
{
    return __int_as_float(m_shr(__float_as_int(v), __float_as_int(old)));
}
__device__ __forceinline__ double m_shr(double v, double old)
{
    const long long b = __double_as_longlong(v), o = __double_as_longlong(old);
    const int lo = m_shr((int)(b & 0xffffffffll), (int)(o & 0xffffffffll));
    const int hi = m_shr((int)(b >> 32), (int)(o >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// until *p >= need; bounded (then the launch is marked and every wait of
// the workgroup falls through, so that it drains)
template<class T>
__device__ __forceinline__ void m_wait(const int* p, int need, MarchShared<T>& S,
                                       unsigned int* err, DevState* st)
{
    uint32_t spins = 0;
#pragma unroll 1
    while (m_ld(p) < need)
    {
        if (m_ld(&S.expired)) break;
        if (++spins > M_LDS_SPINS)
        {
            m_st(&S.expired, 1);
            *err = 1;
            if (st) st->scheduleError = 1;
            break;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    asm volatile("" ::: "memory");
}

template<class T, int MODE>
__device__ __forceinline__ void march_compute(const MarchArgs<T>& A, MarchShared<T>& S,
                                              int pencil, int v, int lane, DevState* st)
{
    typedef typename MBits<T>::V2 V2;
    constexpr int NA = MarchMode<MODE>::na, NO = MarchMode<MODE>::no, MD = MarchMode<MODE>::md;
    const int il = lane & 15, jl = lane >> 4;
    const V2* cp = reinterpret_cast<const V2*>(A.coef)
                   + (int64_t)(pencil*MW + v)*A.nB*(2*NA*64) + lane;
    const V2* op = reinterpret_cast<const V2*>(A.old)
                   + (int64_t)(pencil*MW + v)*A.nB*(2*NO*64) + lane;
    V2 cb[MD][2][NA];
    V2 ob[MD][2][NO > 0 ? NO : 1];
#pragma unroll
    for (int u = 0; u < MD; u++)
    {
#pragma unroll
        for (int q = 0; q < 2*NA; q++) cb[u][q/NA][q % NA] = cp[(u*2*NA + q)*64];
#pragma unroll
        for (int q = 0; q < 2*NO; q++) ob[u][q/(NO ? NO : 1)][q % (NO ? NO : 1)] = op[(u*2*NO + q)*64];
        asm volatile("" ::: "memory");      // in the loop's order
    }
    // The j-1 value of step s: two steps back in the row before (16 lanes
    // down), for the first row the previous wavefront's last row, 6 steps
    // ahead in its count, or the j halo.
    const T* const baseJ = jl > 0 ? &S.ring[v][0][lane - 16]
                         : v > 0 ? &S.ring[v - 1][0][48 + il] : &S.haloJ[0][il];
    const int dJ = jl > 0 ? MRS - 2 : v > 0 ? 6 : 0;
    const int strideJ = jl > 0 || v > 0 ? 64 : MC;
    auto atJ = [&](int s) -> const T* { return baseJ + ((s + dJ) & (MRS - 1))*strideJ; };
    // A block of steps needs its planes staged and the previous wavefront 7
    // steps further than the block's last.
    const int* upStep = v > 0 ? &S.cStep[v - 1] : &S.steps;
    const int steps = A.nB*MG;
    auto upNeed = [&](int b) { return min(MG*b + MG + 6, steps); };
    T* own = &S.ring[v][0][lane];
    const T* hcol = &S.haloI[0][MW*v + jl];
    T prev = T(0);
    m_wait(&S.inReady[v], 1, S, A.err, st);
    m_wait(upStep, upNeed(0), S, A.err, st);
    T nA = own[0], nJ = *atJ(0), nH = hcol[0];
    for (int b0 = 0; b0 < A.nB; b0 += MD)
    {
        // the rings' rows of these MD blocks of steps and of the next ones
        T* const o0 = own + ((b0*MG) & (MRS - 1))*64;
        const T* const h0 = hcol + ((b0*MG) & (MRS - 1))*MC;
        const T* const o1 = own + (((b0 + MD)*MG) & (MRS - 1))*64;
        const T* const h1 = hcol + (((b0 + MD)*MG) & (MRS - 1))*MC;
#pragma unroll
        for (int u = 0; u < MD; u++)
        {
            const int b = b0 + u;
            bool ready = true;
            int seenIn = 0, seenUp = 0;
#pragma unroll
            for (int g = 0; g < MG; g++)
            {
                const int q = u*MG + g, s = b0*MG + q;
                const T a = nA, vJ = nJ, hI = nH;
                auto readNext = [&]
                {
                    nJ = *atJ(s + 1);
                    nA = q + 1 < MD*MG ? o0[(q + 1)*64] : o1[0];
                    nH = q + 1 < MD*MG ? h0[(q + 1)*MC] : h1[0];
                };
                if (g < MG - 1)
                {
                    // what the next block waits for, looked at a step ahead
                    if (g == MG - 2)
                    {
                        seenIn = m_ld(&S.inReady[v]);
                        seenUp = m_ld(upStep);
                    }
                    readNext();
                }
                else
                {
                    ready = __builtin_amdgcn_readfirstlane(seenUp >= upNeed(b + 1)
                                                           && seenIn > b + 1) != 0;
                    asm volatile("" ::: "memory");
                    if (ready) readNext();
                }
                // the reads are under way before the step's arithmetic
                __builtin_amdgcn_sched_barrier(0);
                const T vI = m_shr(prev, hI);
                const V2* c = cb[u][g >> 1];
                auto comp = [&](const V2& t) { return (g & 1) ? t.y : t.x; };
                T w;
                if constexpr (MODE == MARCH_GS_FWD)
                {
                    // lower products k, j, i of new values, then the upper
                    // ones i, j, k of old values
                    const V2* o = ob[u][g >> 1];
                    w = a - comp(c[0])*prev;
                    w = w - comp(c[1])*vJ;
                    w = w - comp(c[2])*vI;
                    w = w - comp(o[0]);
                    w = w - comp(o[1]);
                    w = w - comp(o[2]);
                    w = w/comp(c[3]);
                }
                else if constexpr (MODE == MARCH_GS_BWD)
                {
                    // a: the source less the lower products; upper ones i, j, k
                    w = a - comp(c[2])*vI;
                    w = w - comp(c[1])*vJ;
                    w = w - comp(c[0])*prev;
                    w = w/comp(c[3]);
                }
                else
                {
                    w = MODE == MARCH_BWD ? a : comp(c[0])*a;
                    w = w - comp(c[NA - 3])*prev;
                    w = w - comp(c[NA - 2])*vJ;
                    w = w - comp(c[NA - 1])*vI;
                }
                o0[q*64] = w;
                prev = w;
                if (g == MG - 1)
                {
                    // (a wavefront's LDS accesses complete in order: the
                    // results are in the ring before the count)
                    asm volatile("" ::: "memory");
                    if (lane == 0) m_st(&S.cStep[v], s + 1);
                    // (always the same number of accesses: a branch around
                    // them would make the compiler wait for later blocks'
                    // loads as well)
                    const V2* cn = cp + (int64_t)min(b + MD, A.nB - 1)*(2*NA*64);
#pragma unroll
                    for (int e = 0; e < 2*NA; e++) cb[u][e/NA][e % NA] = cn[e*64];
                    if constexpr (NO > 0)
                    {
                        const V2* on = op + (int64_t)min(b + MD, A.nB - 1)*(2*NO*64);
#pragma unroll
                        for (int e = 0; e < 2*NO; e++) ob[u][e/NO][e % NO] = on[e*64];
                    }
                    asm volatile("" ::: "memory");
                    if (!ready && b + 1 < A.nB)
                    {
                        m_wait(&S.inReady[v], b + 2, S, A.err, st);
                        m_wait(upStep, upNeed(b + 1), S, A.err, st);
                        readNext();
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

// Input wavefront v: the planes of its four rows into the ring, with the
// halos of the pencils upstream, and (backward) the sum of w*dotR over the
// finished planes.  Offsets run on by one addition; what lies outside the
// box lies outside the buffer (a negative offset wraps there) and reads 0.
template<class T, int MODE>
__device__ __forceinline__ double march_input(const MarchArgs<T>& A, MarchShared<T>& S,
                                              int pencil, int v, int lane, int nAct,
                                              DevState* st)
{
    typedef typename MBits<T>::U U;
    typedef MBits<T> M;
    constexpr bool BWD = MarchMode<MODE>::bwd, DOT = MODE == MARCH_BWD;
    constexpr U SENT = M::sent;
    constexpr unsigned int sT = sizeof(T);
    // input and halo blocks in flight (what the registers hold; MLAG is a
    // multiple of it where the sum is taken)
    constexpr int MH = DOT ? 3 : 6;
    constexpr unsigned int HB = MG*MC*sT;       // a halo block
    const int PI = pencil % A.nPI, PJ = pencil/A.nPI;
    const int il = lane & 15, jl = lane >> 4;
    const int i = PI*MC + il, j = PJ*MC + MW*v + jl;
    const bool col = i < A.nx && j < A.ny;
    const unsigned int sz = (unsigned int)A.nx*A.ny, szB = sz*sT;
    const unsigned int step = BWD ? 0u - szB : szB;     // from plane to plane
    const unsigned int plane0 = BWD ? (A.nz - 1)*szB : 0u;
    const unsigned int cxy = col ? plane0 + (BWD ? sz - 1 - (i + A.nx*j) : i + A.nx*j)*sT : M_OOB;
    const unsigned int dxy = col ? step : 0u;
    const unsigned int bytes = szB*(unsigned int)A.nz;
    const bool dot = DOT && A.dotR != nullptr;
    const __amdgpu_buffer_rsrc_t rX = m_rsrc(A.x, bytes);
    const __amdgpu_buffer_rsrc_t rR = m_rsrc(dot ? A.dotR : A.x, dot ? bytes : 0);
    // this pencil's halo slots, by the step that reads them: i halo 4 steps
    // x 4 rows in lanes 0..15, j halo (first wavefront) 4 steps x 16 columns
    const int hk = (lane >> 2) & 3, hr = lane & 3;
    const int64_t hSlots = (int64_t)(A.nz + MC)*MC;
    const __amdgpu_buffer_rsrc_t rI = m_rsrc(A.halo + pencil*hSlots,
                                             PI > 0 ? (A.nz + MSKI)*MC*sT : 0);
    const __amdgpu_buffer_rsrc_t rJ =
        m_rsrc(A.halo + ((int64_t)pencil + A.nPI*A.nPJ)*hSlots,
               PJ > 0 && v == 0 ? (A.nz + MSKJ)*MC*sT : 0);
    unsigned int vI = lane < 16 && PJ*MC + MW*v + hr < A.ny ? (hk*MC + MW*v + hr)*sT : M_OOB;
    unsigned int vJ = i < A.nx ? (jl*MC + il)*sT : M_OOB;
    // LDS places: the lane's column at the step of plane 4 B, the halo rows
    char* const ring = (char*)&S.ring[v][0][lane];
    char* const ringI = (char*)&S.haloI[0][MW*v + hr];
    char* const ringJ = (char*)&S.haloJ[0][il];
    constexpr unsigned int RM = MRS*64*sT - 1, HM = MRS*MC*sT - 1;
    unsigned int tX = (il + 2*jl)*64*sT, tI = hk*MC*sT, tJ = jl*MC*sT;
    U xr[MH][MG], rr[DOT ? MH : 1][MG];
    U hI[MH], hJ[MH], sI = SENT, sJ = SENT;
    // (dotR runs MLAG blocks behind: it starts before the first plane)
    unsigned int vX = cxy, vR = cxy - MG*MLAG*dxy;
    // Every access of the loop is issued on every turn, and the entry
    // issues them in the same order: with a branch around one the compiler
    // could not count the accesses in flight and would wait for later
    // blocks' loads.
    auto loadX = [&](U (&r)[MG])
    {
#pragma unroll
        for (int g = 0; g < MG; g++)
        {
            r[g] = M::template load<0>(rX, vX, 0);
            vX += dxy;
        }
    };
    auto loadR = [&](U (&r)[MG])
    {
#pragma unroll
        for (int g = 0; g < MG; g++)
        {
            r[g] = M::template load<0>(rR, vR, 0);
            vR += dxy;
        }
    };
#pragma unroll
    for (int u = 0; u < MH; u++)
    {
        if constexpr (DOT) loadR(rr[u]);
        asm volatile("" ::: "memory");
        M::template store<M_COH>(rI, 0, M_OOB, 0);
        M::template store<M_COH>(rJ, 0, M_OOB + 8, 0);
        asm volatile("" ::: "memory");
        loadX(xr[u]);
        hI[u] = M::template load<M_COH>(rI, vI + u*HB, 0);
        hJ[u] = M::template load<M_COH>(rJ, vJ + u*HB, 0);
        asm volatile("" ::: "memory");
    }
    double acc = 0.0;
    const int total = (A.nPB + MLAG + MH - 1)/MH*MH;
    const int* const next = v + 1 < nAct ? &S.cStep[v + 1] : &S.steps;
    for (int B0 = 0; B0 < total; B0 += MH)
    {
#pragma unroll
        for (int u = 0; u < MH; u++)
        {
            const int B = B0 + u;
            // The ring slots of block B are free once block B - 16 is
            // written and read by the next wavefront; planes 4 (B - 12)
            // .. +3 are finished (their last lane is 21 steps behind).
            const int needC = MG*min(B - 5, A.nB), needO = MG*min(B - 9, A.nB);
            const int needN = MG*min(B - 11, A.nB);
            const int seenO = m_ld(&S.oStep[v]), seenN = m_ld(next);
            if constexpr (DOT)
            {
                const int seenC = m_ld(&S.cStep[v]);
                asm volatile("" ::: "memory");
                if (seenC < needC) m_wait(&S.cStep[v], needC, S, A.err, st);
                T val[MG];
#pragma unroll
                for (int g = 0; g < MG; g++)
                    val[g] = *(const T*)(ring + ((tX + (MRS - MG*MLAG + g)*64*sT) & RM));
#pragma unroll
                for (int g = 0; g < MG; g++) acc += (double)val[g]*(double)M::val(rr[u][g]);
                loadR(rr[u]);
            }
            asm volatile("" ::: "memory");
            if (__builtin_amdgcn_readfirstlane(seenO < needO || seenN < needN))
            {
                m_wait(&S.oStep[v], needO, S, A.err, st);
                m_wait(next, needN, S, A.err, st);
            }
#pragma unroll
            for (int g = 0; g < MG; g++)
                *(T*)(ring + ((tX + g*64*sT) & RM)) = M::val(xr[u][g]);
            // a slot whose producer was not there yet when the block was
            // sampled; sI, sJ: a later sample, from the last block's polling
            U cI = hI[u], cJ = hJ[u];
            cI = cI == SENT ? sI : cI;
            cJ = cJ == SENT ? sJ : cJ;
            sI = sJ = SENT;
            uint32_t spins = 0;
#pragma unroll 1
            while (__any(cI == SENT || cJ == SENT))
            {
                if (m_ld(&S.expired)) break;
                if (++spins > M_GLOBAL_SPINS)
                {
                    m_st(&S.expired, 1);
                    *A.err = 1;
                    if (st) st->scheduleError = 1;
                    break;
                }
                // this block and the next, so that a producer just ahead is
                // followed block by block
                asm volatile("" ::: "memory");
                const U t0 = M::template load<M_COH>(rI, vI, 0);
                const U t1 = M::template load<M_COH>(rJ, vJ, 0);
                sI = M::template load<M_COH>(rI, vI + HB, 0);
                sJ = M::template load<M_COH>(rJ, vJ + HB, 0);
                cI = cI == SENT ? t0 : cI;
                cJ = cJ == SENT ? t1 : cJ;
                // the samples have arrived (nothing of the polling is in
                // flight where the paths meet)
                asm volatile("" : "+v"(cI), "+v"(cJ), "+v"(sI), "+v"(sJ));
            }
            if (lane < 16) *(T*)(ringI + (tI & HM)) = M::val(cI);
            if (v == 0) *(T*)(ringJ + (tJ & HM)) = M::val(cJ);
            M::template store<M_COH>(rI, SENT, vI, 0);
            M::template store<M_COH>(rJ, SENT, vJ, 0);
            asm volatile("" ::: "memory");
            if (lane == 0) m_st(&S.inReady[v], B + 1);
            loadX(xr[u]);
            hI[u] = M::template load<M_COH>(rI, vI + MH*HB, 0);
            hJ[u] = M::template load<M_COH>(rJ, vJ + MH*HB, 0);
            asm volatile("" ::: "memory");
            vI += HB;
            vJ += HB;
            tX += MG*64*sT;
            tI += MG*MC*sT;
            tJ += MG*MC*sT;
        }
    }
    return acc;
}

// Output wavefront v: publishes the boundary values of its rows to the
// pencils downstream as each block of steps is done, and writes the planes
// that the block finished.  It waits on LDS only, never on memory.
template<class T, bool BWD>
__device__ __forceinline__ void march_output(const MarchArgs<T>& A, MarchShared<T>& S,
                                             int pencil, int v, int lane, DevState* st)
{
    typedef MBits<T> M;
    constexpr unsigned int sT = sizeof(T);
    const int PI = pencil % A.nPI, PJ = pencil/A.nPI;
    const int il = lane & 15, jl = lane >> 4;
    const int i = PI*MC + il, j = PJ*MC + MW*v + jl;
    const bool col = i < A.nx && j < A.ny;
    const unsigned int sz = (unsigned int)A.nx*A.ny, szB = sz*sT;
    const unsigned int step = BWD ? 0u - szB : szB;
    // the first block ends with plane -18
    unsigned int vW = (BWD ? (A.nz - 1 + MSKEW)*szB + (sz - 1 - (i + A.nx*j))*sT
                           : (i + A.nx*j)*sT - MSKEW*szB);
    const __amdgpu_buffer_rsrc_t rW = m_rsrc(A.w, szB*(unsigned int)A.nz);
    // a block's boundary values: the column beside the next pencil along i
    // in lanes 0..15 (step lane >> 2, row lane & 3), the row beside the next
    // pencil along j (last wavefront; step jl, column il).  Step s makes
    // what the reader's step s - 15 (i) or s - 6 (j) takes; steps that it
    // does not have lie outside its slots.
    const int64_t hSlots = (int64_t)(A.nz + MC)*MC;
    const __amdgpu_buffer_rsrc_t rI = m_rsrc(A.halo + ((int64_t)pencil + 1)*hSlots,
                                             PI + 1 < A.nPI ? (A.nz + MSKI)*MC*sT : 0);
    const bool lastRow = v == MW - 1 && PJ + 1 < A.nPJ;
    const __amdgpu_buffer_rsrc_t rJ =
        m_rsrc(A.halo + ((int64_t)pencil + A.nPI + A.nPI*A.nPJ)*hSlots,
               lastRow ? (A.nz + MSKJ)*MC*sT : 0);
    const int gI = (lane >> 2) & 3, rw = lane & 3;
    unsigned int vI = lane < 16 && PJ*MC + MW*v + rw < A.ny
                      ? ((gI - 15)*MC + MW*v + rw)*sT : M_OOB;
    unsigned int vJ = i < A.nx ? ((jl - 6)*MC + il)*sT : M_OOB;
    const char* const ring = (const char*)&S.ring[v][0][lane];
    const char* const srcI = (const char*)&S.ring[v][0][16*rw + 15];
    const char* const srcJ = (const char*)&S.ring[v][0][48 + il];
    constexpr unsigned int RM = MRS*64*sT - 1, RB = 64*sT;
    unsigned int tW = (il + 2*jl - MSKEW)*RB, tI = gI*RB, tJ = jl*RB;
    const int steps = A.nB*MG;
    for (int s = 0; s < steps; s += MG)
    {
        m_wait(&S.cStep[v], s + MG, S, A.err, st);
        const T bI = *(const T*)(srcI + (tI & RM));
        const T bJ = *(const T*)(srcJ + (tJ & RM));
        T val[MG];
#pragma unroll
        for (int g = 0; g < MG; g++) val[g] = *(const T*)(ring + ((tW + g*RB) & RM));
        M::template store<M_COH>(rI, M::bits(bI), vI, 0);
        if (lastRow) M::template store<M_COH>(rJ, M::bits(bJ), vJ, 0);
        if (col)
#pragma unroll
            for (int g = 0; g < MG; g++)
                M::template store<0>(rW, M::bits(val[g]), vW + g*step, 0);
        // (the values are read before the count: the stores wait for them)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (lane == 0) m_st(&S.oStep[v], s + MG);
        vW += MG*step;
        vI += MG*MC*sT;
        vJ += MG*MC*sT;
        tW += MG*RB;
        tI += MG*RB;
        tJ += MG*RB;
    }
}

template<class T, int MODE>
__global__ __launch_bounds__(3*MW*64)
void k_sweep_march(MarchArgs<T> A, DevState* st, FusedFinalize F)
{
    __shared__ __align__(16) MarchShared<T> S;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nP = A.nPI*A.nPJ;
    if (st && st->done)
    {
        if (tid == 0) atomicAdd(A.ticket, 1ull);      // every launch takes its tickets
        return;
    }
    if (tid == 0)
    {
        // pencil of this ticket: along the diagonals PI + PJ
        int p = -1;
        const unsigned long long t = atomicAdd(A.ticket, 1ull) - A.ticketBase;
        if (t < (unsigned long long)nP)
        {
            int r = (int)t, d = 0;
            for (;; d++)
            {
                const int lo = max(0, d - A.nPJ + 1), hi = min(d, A.nPI - 1);
                const int len = hi - lo + 1;
                if (r < len) { p = (lo + r) + A.nPI*(d - lo - r); break; }
                r -= len;
            }
        }
        else
        {
            *A.err = 1;
            if (st) st->scheduleError = 1;
        }
        S.pencil = p;
        S.expired = 0;
        S.steps = A.nB*MG;
        for (int q = 0; q < MW; q++) { S.inReady[q] = 0; S.cStep[q] = S.oStep[q] = 0; S.dot[q] = 0.0; }
    }
    // (ring and halos are adjacent)
    for (int q = tid; q < (int)(sizeof(T)*MRS*(MW*64 + 2*MC)/16); q += 3*MW*64)
        reinterpret_cast<uint4*>(S.ring)[q] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    const int pencil = __builtin_amdgcn_readfirstlane(S.pencil);
    if (pencil < 0) return;
    const int PJ = pencil/A.nPI;
    const int nAct = min(MW, (A.ny - PJ*MC + 3) >> 2);
    const int v = __builtin_amdgcn_readfirstlane(wave & (MW - 1));
    if (v < nAct)
    {
        const int role = __builtin_amdgcn_readfirstlane(wave/MW);
        if (role == 0)
        {
            __builtin_amdgcn_s_setprio(3);
            march_compute<T, MODE>(A, S, pencil, v, lane, st);
            __builtin_amdgcn_s_setprio(0);
        }
        else if (role == 1)
        {
            __builtin_amdgcn_s_setprio(2);
            march_output<T, MarchMode<MODE>::bwd>(A, S, pencil, v, lane, st);
            __builtin_amdgcn_s_setprio(0);
        }
        else
        {
            double acc = march_input<T, MODE>(A, S, pencil, v, lane, nAct, st);
            if constexpr (MODE == MARCH_BWD)
            {
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
                if (lane == 0) S.dot[v] = acc;
            }
        }
    }
    if constexpr (MODE == MARCH_BWD)
    {
        if (A.dotR == nullptr) return;
        __syncthreads();
        double acc = 0.0;
        if (tid == 0)
            for (int q = 0; q < MW; q++) acc += S.dot[q];
        partials_arrive(acc, 0.0, A.partials, nP, pencil, F);
    }
}

// Values of one pass in wavefront order: for wavefront (pencil, v), block of
// 4 steps, pair of steps and value q, lane's two values.  DIC / DILU passes:
// rD (forward) and the three coefficients times it; Gauss-Seidel: the
// coefficients and the diagonal (rD); OLD: the coefficients times rD (psi)
// at the neighbour on the other side.
// A workgroup writes one value of 64 steps of one wavefront: it reads the
// planes these steps touch as rows of 16 cells and turns them into steps in
// LDS.  (Read in step order every lane is in another plane: with that the
// products of a 256^3 forward sweep took longer than the sweep.)
constexpr int MPS = 64;           // steps per workgroup
template<class T, int MODE, bool OLD>
__global__ __launch_bounds__(256)
void k_march_pack(int nx, int ny, int nz, int nPI, int nB, const T* __restrict__ rD,
                  const T* __restrict__ dK, const T* __restrict__ dJ, const T* __restrict__ dI,
                  int shift, typename MBits<T>::V2* __restrict__ out, const DevState* st)
{
    typedef typename MBits<T>::V2 V2;
    constexpr bool BWD = MarchMode<MODE>::bwd, GS = MarchMode<MODE>::gs;
    constexpr int NA = OLD ? MarchMode<MODE>::no : MarchMode<MODE>::na;
    __shared__ T buf[MPS][64];
    if (st && st->done) return;
    const int wv = blockIdx.x, pencil = wv/MW, v = wv % MW;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int PI = pencil % nPI, PJ = pencil/nPI;
    const int il = lane & 15, jl = lane >> 4;
    const int i = PI*MC + il, j = PJ*MC + MW*v + jl;
    if (PJ*MC + MW*v >= ny) return;
    const bool col = i < nx && j < ny;
    const int64_t sy = nx, sz = (int64_t)nx*ny, last = sz*nz - 1;
    const int s0 = blockIdx.y*MPS, s1 = min(s0 + MPS, nB*MG);
    // value q: the product or coefficient of direction e (k, j, i), or the
    // factor itself
    const int q = blockIdx.z;
    const int e = OLD ? 2 - q : GS ? q : q - (NA - 3);
    const bool factor = e < 0 || e > 2;
    const T* const dir = e == 2 ? dI : e == 1 ? dJ : dK;
    const int64_t off = e == 2 ? 1 : e == 1 ? sy : sz;
    const bool inPlane = OLD ? (e == 2 ? i < nx - 1 : e == 1 ? j < ny - 1 : true)
                             : (e == 2 ? i > 0 : e == 1 ? j > 0 : true);
    const bool use = col && (factor || inPlane);
    const int kLo = !OLD && e == 0 ? 1 : 0, kHi = OLD && e == 0 ? nz - 1 : nz;
#pragma unroll 8
    for (int k = s0 - MSKEW + wave; k < s1; k += 4)
    {
        const bool ok = use && k >= kLo && k < kHi;
        const int64_t cf = ok ? i + sy*j + sz*k : 0;
        const int64_t c = BWD ? last - cf : cf;
        T t;
        if (factor) t = ok ? rD[c] : T(GS ? 1 : 0);
        else
        {
            const T a = dir[ok && shift ? c + off : c];
            if constexpr (OLD) t = a*rD[ok ? c + off : c];
            else if constexpr (GS) t = a;
            else t = rD[c]*a;
            t = ok ? t : T(0);
        }
        const int s = k + il + 2*jl - s0;
        if (s >= 0 && s < MPS) buf[s][lane] = t;
    }
    __syncthreads();
    for (int h = wave; h < (s1 - s0)/2; h += 4)
        out[((int64_t)wv*nB*2 + s0/2 + h)*NA*64 + q*64 + lane] =
            V2{buf[2*h][lane], buf[2*h + 1][lane]};
}

// The source of the backward Gauss-Seidel rows: b less the lower products
// k, j, i of the forward pass's values (symGaussSeidelSmoother.C:139-183)
template<class T>
__global__ __launch_bounds__(256)
void k_march_prime(int nx, int ny, int nz, const T* b, const T* psi, const T* dK, const T* dJ,
                   const T* dI, T* out, const DevState* st)
{
    if (st && st->done) return;
    const int sy = nx;
    const int64_t sz = (int64_t)nx*ny;
    const int q = blockIdx.x*256 + threadIdx.x;
    if (q >= sz) return;
    const int j = q/nx, i = q - j*nx;
    for (int k = blockIdx.y; k < nz; k += gridDim.y)
    {
        const int64_t c = q + sz*k;
        T t = b[c];
        if (k > 0) t = t - dK[c]*psi[c - sz];
        if (j > 0) t = t - dJ[c]*psi[c - sy];
        if (i > 0) t = t - dI[c]*psi[c - 1];
        out[c] = t;
    }
}

template<class U>
__global__ __launch_bounds__(256)
void k_march_fill(int64_t n, U* a, U v)
{
    for (int64_t q = blockIdx.x*(int64_t)256 + threadIdx.x; q < n; q += (int64_t)gridDim.x*256)
        a[q] = v;
}

static void march_shape(const TileView& G, int32_t& nPI, int32_t& nPJ, int32_t& nPB, int32_t& nB)
{
    nPI = (G.nx + MC - 1)/MC;
    nPJ = (G.ny + MC - 1)/MC;
    nPB = (G.nz + MG - 1)/MG;
    nB = (G.nz + MSKEW + MG - 1)/MG;
    nB = (nB + MD - 1)/MD*MD;
}

template<class T, int MODE, bool OLD>
static void march_pack(const TileView& G, const T* rD, const T* const dir[3], bool dirShift,
                       DBuf<T>& out, const DevState* st, hipStream_t s)
{
    int32_t nPI, nPJ, nPB, nB;
    march_shape(G, nPI, nPJ, nPB, nB);
    const int64_t waves = (int64_t)nPI*nPJ*MW;
    const int nv = OLD ? MarchMode<MODE>::no : MarchMode<MODE>::na;
    out.alloc((size_t)waves*nB*MG*64*nv);
    hipLaunchKernelGGL((k_march_pack<T, MODE, OLD>),
                       dim3((unsigned)waves, (unsigned)((nB*MG + MPS - 1)/MPS), (unsigned)nv),
                       dim3(256), 0, s, G.nx, G.ny, G.nz, nPI, nB, rD, dir[0], dir[1], dir[2],
                       dirShift ? 1 : 0, reinterpret_cast<typename MBits<T>::V2*>(out.p), st);
}

template<class T>
void launch_march_pack(bool backward, const TileView& G, const T* rD, const T* const dir[3],
                       bool dirShift, MarchBufs<T>& b, hipStream_t s)
{
    if (backward) march_pack<T, MARCH_BWD, false>(G, rD, dir, dirShift, b.bwd, nullptr, s);
    else march_pack<T, MARCH_FWD, false>(G, rD, dir, dirShift, b.fwd, nullptr, s);
}

void launch_march_pack_gs(bool backward, const TileView& G, const double* diag,
                          const double* const dir[3], bool dirShift, MarchBufs<double>& b,
                          hipStream_t s)
{
    if (backward)
        march_pack<double, MARCH_GS_BWD, false>(G, diag, dir, dirShift, b.gsBwd, nullptr, s);
    else march_pack<double, MARCH_GS_FWD, false>(G, diag, dir, dirShift, b.gsFwd, nullptr, s);
}

template<class T>
void march_prepare_halo(const TileView& G, MarchBufs<T>& b, hipStream_t s)
{
    typedef typename MBits<T>::U U;
    if (b.haloReady) return;
    int32_t nPI, nPJ, nPB, nB;
    march_shape(G, nPI, nPJ, nPB, nB);
    const int64_t n = 2*(int64_t)nPI*nPJ*(G.nz + MC)*MC;
    b.halo.alloc((size_t)n);
    const unsigned grid = (unsigned)std::min<int64_t>((n + 255)/256, 2048);
    hipLaunchKernelGGL((k_march_fill<U>), dim3(grid), dim3(256), 0, s, n,
                       reinterpret_cast<U*>(b.halo.p), MBits<T>::sent);
    b.haloReady = true;
}

template<class T>
static MarchArgs<T> march_args(const TileView& G, const MarchBufs<T>& b, const TileSync& sync,
                               unsigned int* err)
{
    if (!b.haloReady) fail(FH_ERR_INVALID, "internal: marching sweep without its halos");
    MarchArgs<T> A{};
    A.nx = G.nx; A.ny = G.ny; A.nz = G.nz;
    march_shape(G, A.nPI, A.nPJ, A.nPB, A.nB);
    A.halo = b.halo.p;
    A.ticket = sync.ticket;
    A.ticketBase = sync.ticketBase;
    A.err = err;
    return A;
}

template<class T, int MODE>
static int32_t march_launch(const MarchArgs<T>& A, TileSync& sync, DevState* st, hipStream_t s,
                            const FusedFinalize& F = FusedFinalize())
{
    const int32_t nP = A.nPI*A.nPJ;
    hipLaunchKernelGGL((k_sweep_march<T, MODE>), dim3(nP), dim3(3*MW*64), 0, s, A, st, F);
    sync.ticketBase += (unsigned long long)nP;
    sync.epoch++;
    return nP;
}

template<class T>
int32_t launch_sweep_march(bool backward, const TileView& G, const SweepData<T>& d,
                           const MarchBufs<T>& b, TileSync& sync, unsigned int* err,
                           DevState* st, hipStream_t s, const FusedFinalize& F)
{
    if (!b.fwd.p || !b.bwd.p)
        fail(FH_ERR_INVALID, "internal: marching sweep without its buffers");
    if (d.dotR && (!backward || !d.partials))
        fail(FH_ERR_INVALID, "internal: fused sum on a sweep that does not provide it");
    MarchArgs<T> A = march_args<T>(G, b, sync, err);
    A.coef = backward ? b.bwd.p : b.fwd.p;
    A.x = backward ? d.w : d.x;
    A.w = d.w;
    A.dotR = backward ? d.dotR : nullptr;
    A.partials = d.partials;
    return backward ? march_launch<T, MARCH_BWD>(A, sync, st, s, F)
                    : march_launch<T, MARCH_FWD>(A, sync, st, s, F);
}

void launch_sweep_march_gs(bool backward, const TileView& G, const SweepData<double>& d,
                           MarchBufs<double>& b, TileSync& sync, unsigned int* err,
                           DevState* st, hipStream_t s)
{
    MarchArgs<double> A = march_args<double>(G, b, sync, err);
    A.w = d.w;
    if (!backward)
    {
        march_pack<double, MARCH_GS_FWD, true>(G, d.w, d.dir, d.dirShift != 0, b.gsOld, st, s);
        A.coef = b.gsFwd.p;
        A.old = b.gsOld.p;
        A.x = d.x;
        march_launch<double, MARCH_GS_FWD>(A, sync, st, s);
        return;
    }
    const int64_t sz = (int64_t)G.nx*G.ny;
    b.gsPrime.alloc((size_t)(sz*G.nz));
    const unsigned gx = (unsigned)((sz + 255)/256);
    const unsigned gy = (unsigned)std::max<int64_t>(1, std::min<int64_t>(G.nz, 4096/gx));
    hipLaunchKernelGGL((k_march_prime<double>), dim3(gx, gy), dim3(256), 0, s, G.nx, G.ny, G.nz,
                       d.x, d.w, d.dir[0], d.dir[1], d.dir[2], b.gsPrime.p, st);
    A.coef = b.gsBwd.p;
    A.x = b.gsPrime.p;
    march_launch<double, MARCH_GS_BWD>(A, sync, st, s);
}

#define MARCH_INST(T) \
template void launch_march_pack<T>(bool, const TileView&, const T*, const T* const[3], bool, \
                                   MarchBufs<T>&, hipStream_t); \
template void march_prepare_halo<T>(const TileView&, MarchBufs<T>&, hipStream_t); \
template int32_t launch_sweep_march<T>(bool, const TileView&, const SweepData<T>&, \
                                       const MarchBufs<T>&, TileSync&, unsigned int*, DevState*, \
                                       hipStream_t, const FusedFinalize&);
MARCH_INST(double)
MARCH_INST(float)

} // namespace fh
