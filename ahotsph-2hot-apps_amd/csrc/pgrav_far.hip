// The far cells of every sink group through a local expansion (pgrav_local.h).
//
// One wave per group.  It scans the group's cell lists 64 entries at a time: the far
// entries (pgrav_far.h) queue in LDS, the others go, in list order, to the list that the
// pair kernel reads instead of the group's own.  Whenever the queue holds an entry for
// every lane, each lane takes one cell: it gathers the cell's record and adds the
// cell's expansion to its own 81 (softened: 101) coefficients in registers.  The lanes'
// coefficients meet through LDS in a fixed order, and their sum is evaluated at the
// group's sinks into a buffer of its own, from where the pair kernel takes it up: the
// result array only ever holds whole results, so that a reader of the last evaluation's
// on another stream sees the same values while the next one of the same bodies runs.
//
// Bound by VALU at two waves per SIMD: 1,500 instructions per 64 order-4 cells (1,050
// order 2, 345 order 0) against 110 (45, 16) x 64 in pairs, ~110 per 64 entries scanned
// and ~2,300 per group.  Clustered 16.8 M: 7.0 ms, which take 62 % of the order-4 cells
// out of the pair kernel, 42.5 -> 20 ms.
#include <math.h>

#include "pgrav_batch.h"
#include "pgrav_device.h"
#include "pgrav_far.h"
#include "pgrav_local.h"

namespace pgrav {

namespace {

struct FarArgs {
    const double4 *__restrict__ bpos, *__restrict__ cpos;
    const float *__restrict__ mom;
    const int64_t *__restrict__ gfirst;
    const int *__restrict__ gcount;
    const int64_t *__restrict__ gslot_off;
    const uint32_t *__restrict__ gslot;
    const double4 *__restrict__ gcen;
    const int64_t *__restrict__ off;
    const uint32_t *__restrict__ idx;
    const uint8_t *__restrict__ img;
    int img_f, ngroups;
    double eps, box, ibox, ewratio;
    double *__restrict__ far2;
    uint32_t *__restrict__ near;  // the entries left to the pair kernel, at their list's start
    uint8_t *__restrict__ near_img;
    int *__restrict__ near_n;  // [3][ngroups]
    float4 *__restrict__ pull;  // [n][2]
};

constexpr int ROWS = 16;  // coefficients summed over the lanes per LDS round

struct FarShared {
    float4 off[128];  // queued entries: offset and mass
    uint32_t node[128];
    double low[4];  // degrees 0 and 1, the bulk of the pull, summed in FP64
    float red[ROWS][65];
    float sum[LX_ALL];
};

template <int ORDER, bool SOFT>
__device__ __forceinline__ void add_queued(const FarArgs &A, const FarShared &sh, int at, float eps2,
                                           float lam, float *acc) {
    const float4 o = sh.off[at];
    float rec[46];
    if constexpr (ORDER > 0) {
        const float4 *__restrict__ r = (const float4 *)(A.mom + (size_t)sh.node[at] * PREC4);
        constexpr int last = ORDER == 4 ? 11 : 2;
#pragma unroll
        for (int q = 1; q <= last; q++) {
            const float4 v = r[q];
            rec[4 * q] = v.x;
            rec[4 * q + 1] = v.y;
            if (4 * q + 2 < 46) {
                rec[4 * q + 2] = v.z;
                rec[4 * q + 3] = v.w;
            }
        }
    }
    lx_add_cell<ORDER, SOFT, float>(rec, o.w, o.x, o.y, o.z, eps2, lam, acc);
}

// Workgroup b's group.  Workgroup b runs on XCD b mod NXCD: each XCD takes runs of
// FAR_RUN groups, which are neighbours and share cells in its L2, dealt in turn.  (In the
// pair kernel's slices, which are of equal cost in pairs and not in far cells, the XCDs
// were busy for 78 % of the launch: clustered 16.8 M 27.8 ms with both kernels, 26.7 ms so,
// and 1 M 1.86 and 1.76 ms; runs of 8 and of 128 within 1 % of it; a fixed grid that takes
// its groups by counters from the slices, 27.0 and 1.81.)
constexpr int FAR_RUN = 32;

static __device__ __forceinline__ int group_of(int b, int ngroups) {
    if (b >= ngroups / (NXCD * FAR_RUN) * (NXCD * FAR_RUN))
        return b;
    const int x = b % NXCD, i = b / NXCD;
    return (i / FAR_RUN * NXCD + x) * FAR_RUN + i % FAR_RUN;
}

// (two waves per SIMD: the coefficients and a turned cell take 256 registers, and with
// three the compiler's spills cost more than the third wave gives)
template <bool SOFT, int PER>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_far(FarArgs A) {
    __shared__ FarShared sh;
    const int g = group_of(blockIdx.x, A.ngroups);
    const int lane = threadIdx.x;
    const int64_t G1 = A.ngroups + 1;
    int64_t ncell = 0;
    for (int kind = 0; kind < 3; kind++) ncell += A.off[kind * G1 + g + 1] - A.off[kind * G1 + g];
    const int cnt = A.gcount[g];
    const double4 gc = A.gcen[g];
    const bool live = lane < cnt;
    int64_t slot;
    if (A.gslot)
        slot = A.gslot[A.gslot_off[g] + (live ? lane : 0)];
    else
        slot = A.gfirst[g] + (live ? lane : 0);
    const double4 sp = A.bpos[slot];
    const double sx = sp.x - gc.x, sy = sp.y - gc.y, sz = sp.z - gc.z;
    double rs2 = sx * sx + sy * sy + sz * sz;
    for (int h = 32; h > 0; h >>= 1) rs2 = fmax(rs2, __shfl_xor(rs2, h));
    const double rs = sqrt(rs2);
    // sinks all but at one point, or outside the sphere that says which image they see (moved
    // bodies): no expansion
    const bool off = ncell < FAR_MIN_CELLS || !(rs > FAR_MIN_RADIUS) ||
                     (PER == 1 && rs > gc.w * (1.0 + 1e-9));
    const double far2 = off ? (double)INFINITY
                            : fmax(rs2 / (FAR_RHO * FAR_RHO), SOFT ? A.eps * A.eps / FAR_ETA : 0.0);
    if (lane == 0)
        A.far2[g] = far2;
    if (off)
        return;
    const float lam = (float)rs, eps2 = (float)(A.eps * A.eps);
    float acc[LX_ALL];
    constexpr int NA = SOFT ? LX_ALL : LX_N;
#pragma unroll
    for (int q = 0; q < LX_ALL; q++) acc[q] = 0.f;

    int head = 0, tail = 0;  // entries queued so far, and taken
    const uint64_t below = (1ull << lane) - 1;
    auto scan = [&](int kind, auto order) {
        constexpr int ORDER = decltype(order)::value;
        const int64_t o0 = A.off[kind * G1 + g], o1 = A.off[kind * G1 + g + 1];
        const bool fills = o1 - o0 >= FAR_MIN_LIST;
        int64_t left = o0;
        // the next round's positions and the indices of the one after it load while a
        // round is taken
        const int64_t i0 = o0 + lane;
        uint32_t e1 = i0 < o1 ? A.idx[i0] : 0, e2 = i0 + 64 < o1 ? A.idx[i0 + 64] : 0;
        double4 s1 = make_double4(0, 0, 0, 0);
        if (i0 < o1)
            s1 = entry_position<PER>(A.cpos, e1, A.img, i0, A.img_f, A.box);
        for (int64_t i = i0; i - lane < o1; i += 64) {
            const uint32_t e = e1;
            const double4 s = s1;
            e1 = e2;
            if (i + 64 < o1)
                s1 = entry_position<PER>(A.cpos, e1, A.img, i + 64, A.img_f, A.box);
            if (i + 128 < o1)
                e2 = A.idx[i + 128];
            const double3 d = entry_offset<PER>(s, gc, A.box, A.ibox);
            const bool far = i < o1 && fills && entry_far<PER>(d, far2, gc, A.box, A.ewratio);
            const uint64_t b = __builtin_amdgcn_ballot_w64(far);
            if (far) {
                const int q = (tail + __popcll(b & below)) & 127;
                sh.off[q] = make_float4((float)d.x, (float)d.y, (float)d.z, (float)s.w);
                sh.node[q] = e;
            }
            tail += __popcll(b);
            if (PER != 1) {
                const bool keep = i < o1 && !far;
                const uint64_t k = __builtin_amdgcn_ballot_w64(keep);
                if (keep) {
                    const int64_t at = left + __popcll(k & below);
                    A.near[at] = e;
                    if (PER == 2)
                        A.near_img[at] = A.img[i];
                }
                left += __popcll(k);
            }
            wave_sync();
            if (tail - head >= 64) {
                add_queued<ORDER, SOFT>(A, sh, (head + lane) & 127, eps2, lam, acc);
                head += 64;
                wave_sync();
            }
        }
        if (lane < tail - head)
            add_queued<ORDER, SOFT>(A, sh, (head + lane) & 127, eps2, lam, acc);
        head = tail;
        wave_sync();
        if (PER != 1 && lane == 0)
            A.near_n[kind * A.ngroups + g] = (int)(left - o0);
    };
    scan(0, std::integral_constant<int, 4>{});
    scan(1, std::integral_constant<int, 2>{});
    scan(2, std::integral_constant<int, 0>{});

    // the lanes' sums, 16 coefficients at a time: four lanes add a row's quarters
#pragma unroll
    for (int c = 0; c < NA; c += ROWS) {
#pragma unroll
        for (int r = 0; r < ROWS; r++)
            if (c + r < NA)
                sh.red[r][lane] = acc[c + r];
        wave_sync();
        const int r = lane >> 2, q = lane & 3;
        if (c == 0) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < 16; k++) s += (double)sh.red[r][16 * q + k];
            s = dpp_add<0x4e, 0xf>(dpp_add<0xb1, 0xf>(s));
            if (q == 0 && r < 4)
                sh.low[r] = s;
            else if (q == 0)
                sh.sum[r] = (float)s;
        } else {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < 16; k++) s += sh.red[r][16 * q + k];
            s = dpp_add<0x4e, 0xf>(dpp_add<0xb1, 0xf>(s));
            if (q == 0 && c + r < NA)
                sh.sum[c + r] = s;
        }
        wave_sync();
    }
    if (live) {
        const float il = 1.f / lam;
        float r[4];
        lx_evaluate<SOFT, 2, float>(sh.sum, (float)sx * il, (float)sy * il, (float)sz * il, il, r);
        // degrees 0 and 1: psi = a0 + (a10 z + (a11 x + b11 y) / 2) / lam
        const double *a = sh.low, ild = 1.0 / (double)lam;
        const double gx = 0.5 * a[2] * ild, gy = 0.5 * a[3] * ild, gz = a[1] * ild;
        const double v[4] = {gx + r[0], gy + r[1], gz + r[2],
                             r[3] - (a[0] + gx * sx + gy * sy + gz * sz)};
        const float4 hi = make_float4((float)v[0], (float)v[1], (float)v[2], (float)v[3]);
        A.pull[2 * slot] = hi;
        A.pull[2 * slot + 1] = make_float4((float)(v[0] - hi.x), (float)(v[1] - hi.y),
                                           (float)(v[2] - hi.z), (float)(v[3] - hi.w));
    }
}

}  // namespace

hipError_t launch_far(const BatchView &v, hipStream_t st) {
    if (v.ngroups <= 0)
        return hipSuccess;
    if (v.periodic < 0 || v.periodic > 2 || (v.periodic == 2 && !v.img))
        return hipErrorInvalidValue;
    FarArgs A;
    A.bpos = v.bpos;
    A.cpos = v.cpos;
    A.mom = v.mom32;
    A.gfirst = v.gfirst;
    A.gcount = v.gcount;
    A.gslot_off = v.gslot_off;
    A.gslot = v.gslot;
    A.gcen = v.gcen;
    A.off = v.off;
    A.idx = v.idx;
    A.img = v.img;
    A.img_f = 2 * v.nimage + 1;
    A.ngroups = v.ngroups;
    A.eps = v.eps;
    A.box = v.box;
    A.ibox = 1.0 / v.box;
    A.ewratio = v.ewratio;
    A.far2 = v.far2;
    A.pull = v.far_pull;
    A.near = v.near;
    A.near_img = v.near_img;
    A.near_n = v.near_n;
    const dim3 grid(v.ngroups), block(64);
    const bool soft = v.soft == SOFT_PLUMMER;
#define FAR(P)                                                       \
    if (soft)                                                        \
        hipLaunchKernelGGL((k_far<true, P>), grid, block, 0, st, A); \
    else                                                             \
        hipLaunchKernelGGL((k_far<false, P>), grid, block, 0, st, A)
    if (v.periodic == 1) {
        FAR(1);
    } else if (v.periodic == 2) {
        FAR(2);
    } else {
        FAR(0);
    }
#undef FAR
    return hipGetLastError();
}

}  // namespace pgrav
