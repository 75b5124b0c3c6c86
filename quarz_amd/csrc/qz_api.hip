// C-ABI glue: error reporting, device information, the batched Thomas solver and the sweep entry points.
#include <hip/hip_runtime.h>

#include <cstdio>

#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "qz_chain.hpp"
#include "qz_device.hpp"
#include "qz_internal.hpp"

namespace {
thread_local std::string g_last_error;
}

int qz_fail(int code, const std::string& msg) {
    g_last_error = msg;
    return code;
}
int qz_fail_hip(hipError_t e, const std::string& where) {
    g_last_error = where + ": " + hipGetErrorString(e);
    return QZ_EHIP;
}

extern "C" const char* qz_last_error(void) { return g_last_error.c_str(); }

extern "C" int qz_device_info(char* arch, int arch_len, int* n_cu) {
    int dev = 0;
    QZ_HIP(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    QZ_HIP(hipGetDeviceProperties(&prop, dev));
    if (arch && arch_len > 0) {
        std::strncpy(arch, prop.gcnArchName, static_cast<size_t>(arch_len) - 1);
        arch[arch_len - 1] = 0;
    }
    if (n_cu) *n_cu = prop.multiProcessorCount;
    return QZ_OK;
}

namespace qz {
// Batched Thomas (src/Tridiag.cpp:111-126), every value formed exactly as the reference forms it.  Element i of system
// s sits at s * ss + i * es of a, b, c, d and x; the forward sweep keeps d' in x and c' in the caller's workspace, which
// the backward sweep reads.
typedef double Pair8 __attribute__((ext_vector_type(2), aligned(8)));   // two doubles at any double's address

// Long systems stored row after row (kRows: es = 1), and few systems of any layout: a DPP row of 16 lanes per system, 8
// rows per lane in registers (qz_chain.hpp), so that a lane reads whole cache lines and a sixteenth of the systems that
// one thread each would need fills the chip.  The next block of rows is loaded while one is run.  The reciprocal is
// chain_recip, checked against the division after each block.  Bound by the chain up to 4096 systems, then by its
// repeated steps.
// Row after row: 4096 systems of 513 rows 41 us (2.1 TB/s), where one thread per system, a row at a time, took 412 us;
// 64 systems of 65 rows 6 us (31 us).
template <bool kRows>
__global__ void __launch_bounds__(64) thomas_lanes_kernel(const Real* a, const Real* b, const Real* c, const Real* d,
                                                          Real* x, Real* cpw, int M, int batch, long long ss,
                                                          long long es) {
    constexpr int R = kChainR;
    const int l = threadIdx.x & 15;
    const int s = min(static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x >> 4), batch - 1);
    const long long o = static_cast<long long>(s) * ss;
    const bool own = static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x >> 4) < batch;
    Real* X = x + o;
    const long long cs = kRows ? 1 : batch;   // c' laid out as the systems are
    Real* CP = cpw + (kRows ? static_cast<size_t>(s) * M : static_cast<size_t>(s));
    const int nb = (M + kChainBlock - 1) / kChainBlock;
    // rows i0 .. i0 + R - 1 of p (stride st), those from M on `rest`
    auto load = [&](const Real* p, long long st, int i0, Real rest, Real (&v)[R]) {
        if (kRows && i0 + R <= M) {
#pragma unroll
            for (int r = 0; r < R; r += 2) {
                const Pair8 t = *reinterpret_cast<const Pair8*>(p + i0 + r);
                v[r] = t.x;
                v[r + 1] = t.y;
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = p[min(i0 + r, M - 1) * st];
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (i0 + r >= M) v[r] = rest;
        }
    };
    auto store = [&](Real* p, long long st, int i0, const Real (&v)[R]) {
        if (!own) return;
        if (kRows && i0 + R <= M) {
#pragma unroll
            for (int r = 0; r < R; r += 2) {
                Pair8 t;
                t.x = v[r];
                t.y = v[r + 1];
                *reinterpret_cast<Pair8*>(p + i0 + r) = t;
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (i0 + r < M) p[(i0 + r) * st] = v[r];
        }
    };
    Real av[R], bv[R], cv[R], dv[R], na[R], nbv[R], nc[R], nd[R], cp[R], dp[R];
    auto load_block = [&](int k) {
        const int i0 = k * kChainBlock + l * R;
        load(a + o, es, i0, Real(0), na);
        load(b + o, es, i0, Real(1), nbv);
        load(c + o, es, i0, Real(0), nc);
        load(d + o, es, i0, Real(0), nd);
    };
    load_block(0);
    Real ccar = Real(0), dcar = Real(0);
    for (int k = 0; k < nb; ++k) {
        const int i0 = k * kChainBlock + l * R;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            av[r] = na[r]; bv[r] = nbv[r]; cv[r] = nc[r]; dv[r] = nd[r];
            if (i0 + r == M - 1) cv[r] = Real(0);   // not used
        }
        if (k + 1 < nb) load_block(k + 1);
        if (i0 == 0) {   // row 0: c_0 / b_0 and d_0 / b_0, through (.. - 0 * 0) * (1 / (1 - 0 * 0))
            cv[0] = cv[0] / bv[0];
            dv[0] = dv[0] / bv[0];
            av[0] = Real(0);
            bv[0] = Real(1);
        }
        const int steps = min(16, (M - k * kChainBlock + R - 1) / R);
        Real qc = ccar, qd = dcar;
        auto rows = [&](auto recip) {
            qc = dpp_prev(qc, cp[R - 1]);
            qd = dpp_prev(qd, dp[R - 1]);
            Real pc = qc, pd = qd;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const Real m = recip(bv[r] - av[r] * pc);
                pd = (dv[r] - av[r] * pd) * m;
                pc = cv[r] * m;
                cp[r] = pc;
                dp[r] = pd;
            }
        };
        cp[R - 1] = dp[R - 1] = Real(0);
#pragma unroll 1
        for (int t = 0; t < steps; ++t) rows([](Real v) { return chain_recip(v); });
        bool bad = false;
        Real p = qc;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const Real v = bv[r] - av[r] * p;
            bad = bad || __double_as_longlong(chain_recip(v)) != __double_as_longlong(Real(1) / v);
            p = cp[r];
        }
        if (__ballot(bad ? 1 : 0)) {
            qc = ccar;
            qd = dcar;
            cp[R - 1] = dp[R - 1] = Real(0);
#pragma unroll 1
            for (int t = 0; t < steps; ++t) rows([](Real v) { return Real(1) / v; });
        }
        if (k + 1 < nb) {   // the last block stays in registers
            store(CP, cs, i0, cp);
            store(X, es, i0, dp);
        }
        ccar = dpp_ror(cp[R - 1]);
        dcar = dpp_ror(dp[R - 1]);
    }
    Real car = Real(0);
    for (int k = nb - 1; k >= 0; --k) {
        const int i0 = k * kChainBlock + l * R;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            cv[r] = i0 + r >= M - 1 ? Real(0) : cp[r];   // x_{M-1} = d'_{M-1} - 0 * 0
            dv[r] = i0 + r >= M ? Real(0) : dp[r];
        }
        if (k > 0) {
            load(CP, cs, i0 - kChainBlock, Real(0), cp);
            load(X, es, i0 - kChainBlock, Real(0), dp);
        }
        const int steps = min(16, (M - k * kChainBlock + R - 1) / R);
        Real q = car;
        av[0] = Real(0);
        for (int t = 0; t < steps; t += 2) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                q = dpp_next(q, av[0]);
                Real v = q;
#pragma unroll
                for (int r = R - 1; r >= 0; --r) {
                    v = dv[r] - cv[r] * v;
                    av[r] = v;
                }
            }
        }
        store(X, es, i0, av);
        car = dpp_rol(av[0]);
    }
}

// Any strides: one thread per system, U rows loaded ahead of the U being run; c' element-major.
// Element-major, 513 rows: 32768 systems 218 us (3.1 TB/s), 576 us without the loads ahead.
template <int U>
__global__ void __launch_bounds__(64) thomas_batched_kernel(const Real* a, const Real* b, const Real* c, const Real* d,
                                                            Real* x, Real* cpw, int M, int batch, long long ss,
                                                            long long es) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= batch) return;
    const long long o = static_cast<long long>(s) * ss;
    const Real *A = a + o, *B = b + o, *C = c + o, *D = d + o;
    Real* X = x + o;
    Real* CP = cpw + s;
    Real av[U], bv[U], cv[U], dv[U], na[U], nb[U], nc[U], nd[U];
    auto load = [&](int i0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const long long e = min(i0 + u, M - 1) * es;
            na[u] = A[e]; nb[u] = B[e]; nc[u] = C[e]; nd[u] = D[e];
        }
    };
    Real cp = C[0] / B[0];
    Real dp = D[0] / B[0];
    if (M > 1) load(1);
    CP[0] = cp;
    X[0] = dp;
    for (int i0 = 1; i0 < M; i0 += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) { av[u] = na[u]; bv[u] = nb[u]; cv[u] = nc[u]; dv[u] = nd[u]; }
        if (i0 + U < M) load(i0 + U);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i0 + u < M) {
                const Real m = Real(1) / (bv[u] - av[u] * cp);
                cp = cv[u] * m;
                dp = (dv[u] - av[u] * dp) * m;
                CP[static_cast<size_t>(i0 + u) * batch] = cp;
                X[(i0 + u) * es] = dp;
            }
    }
    Real xn = dp;
    auto load_back = [&](int i0) {   // rows i0, i0 - 1, ...
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = max(i0 - u, 0);
            na[u] = CP[static_cast<size_t>(i) * batch];
            nd[u] = X[i * es];
        }
    };
    if (M > 1) load_back(M - 2);
    for (int i0 = M - 2; i0 >= 0; i0 -= U) {
#pragma unroll
        for (int u = 0; u < U; ++u) { av[u] = na[u]; dv[u] = nd[u]; }
        if (i0 - U >= 0) load_back(i0 - U);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i0 - u >= 0) {
                xn = dv[u] - av[u] * xn;
                X[(i0 - u) * es] = xn;
            }
    }
}
}  // namespace qz

// Up to kThomasLanesMax systems each takes a DPP row, in any layout (element-major, 513 rows: 2048 systems 57 us against
// 100 us for a thread per system, 4096 86 against 98, 8192 166 against 102).  Of more, those stored row after row with
// more than kThomasThreadRows rows do: a wave runs whole blocks of 8 rows per lane and checks them, whatever a system
// has, and a thread per system is faster while its rows lie in a few cache lines.  Row after row, DPP row against thread:
//   10^6 systems of   2 rows 503 us / 19,   9 rows 682 / 193,   17 rows 751 / 693,   18 rows 759 / 896,   33 rows 863 / 1651
//   8192 systems of   2 rows 6.2 us / 5.4,  9 rows 7.1 / 5.8,   17 rows 7.5 / 6.3,   18 rows 7.7 / 7.0,   33 rows 8.9 / 9.8
constexpr int kThomasLanesMax = 4096;
constexpr int kThomasThreadRows = 17;
// Rows a thread loads ahead: two for systems that have no more after the first, where eight would be loads of the last
// row (2 rows, 4 x 10^6 systems row after row: 89 us, 146 us with eight).
constexpr int kThomasTinyRows = 3;

extern "C" size_t qz_tridiag_workspace_doubles(int M, int batch) {
    return (M < 1 || batch < 1) ? 0 : static_cast<size_t>(M) * static_cast<size_t>(batch);
}

extern "C" int qz_tridiag_thomas_batched(const double* a, const double* b, const double* c, const double* d, double* x,
                                         int M, int batch, long long sys_stride, long long elem_stride, double* work,
                                         void* stream) {
    if (M < 1 || batch < 0) return qz_fail(QZ_EINVAL, "qz_tridiag_thomas_batched: bad extent");
    if (batch == 0) return QZ_OK;
    if (!a || !b || !c || !d || !x || !work) return qz_fail(QZ_EINVAL, "qz_tridiag_thomas_batched: null argument");
    if (elem_stride < 1 || (batch > 1 && sys_stride < 1))
        return qz_fail(QZ_EINVAL, "qz_tridiag_thomas_batched: strides must be positive");
    // systems may interleave (element-major layouts), but no two elements of the batch may share an address:
    // (s, i) and (s + ds, i - di) collide when ds * sys_stride = di * elem_stride with di <= M - 1
    const long long span = (M - 1) * elem_stride + 1;
    if (batch > 1 && sys_stride < span)
        for (long long si = 1; si < batch && si * sys_stride < span; ++si)
            if ((si * sys_stride) % elem_stride == 0)
                return qz_fail(QZ_EINVAL, "qz_tridiag_thomas_batched: strides make two systems overlap");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (batch <= kThomasLanesMax || (elem_stride == 1 && M > kThomasThreadRows)) {
        hipLaunchKernelGGL(elem_stride == 1 ? qz::thomas_lanes_kernel<true> : qz::thomas_lanes_kernel<false>,
                           dim3((batch + 3) / 4), dim3(64), 0, st, a, b, c, d, x, work, M, batch, sys_stride, elem_stride);
        QZ_HIP(hipGetLastError());
        return QZ_OK;
    }
    const int tb = 64;
    hipLaunchKernelGGL(M <= kThomasTinyRows ? qz::thomas_batched_kernel<2> : qz::thomas_batched_kernel<8>,
                       dim3((batch + tb - 1) / tb), dim3(tb), 0, st, a, b, c, d, x, work, M, batch, sys_stride, elem_stride);
    QZ_HIP(hipGetLastError());
    return QZ_OK;
}

extern "C" size_t qz_sweep_workspace_doubles(int M) { return qz_sweep_workspace_doubles_impl(M); }
extern "C" size_t qz_sweep_args_bytes(void) { return sizeof(qz_sweep_args); }

extern "C" int qz_device_tag(char* out, int n) {
    if (!out || n < 1) return qz_fail(QZ_EINVAL, "qz_device_tag: no buffer");
    int dev = 0;
    QZ_HIP(hipGetDevice(&dev));
    hipDeviceProp_t pr;
    QZ_HIP(hipGetDeviceProperties(&pr, dev));
    std::snprintf(out, static_cast<size_t>(n), "%s|%dCU", pr.gcnArchName, pr.multiProcessorCount);
    return QZ_OK;
}

int qz_validate_sweep(const qz_sweep_args& a) {
    if (a.modes != 0 && a.modes != 1) return qz_fail(QZ_EINVAL, "sweep: modes must be 0 or 1");
    if (a.grid.N < 2 || a.grid.N > 2048) return qz_fail(QZ_ERANGE, "sweep: need 2 <= N <= 2048 radial cells");
    if (a.nslices < 1) return qz_fail(QZ_EINVAL, "sweep: nslices < 1");
    if (a.k_begin < 0 || a.k_end < 0 || a.k_end > a.nslices || (a.k_end > 0 && a.k_begin >= a.k_end) ||
        (a.k_end == 0 && a.k_begin >= a.nslices))
        return qz_fail(QZ_EINVAL, "sweep: slice range [k_begin, k_end) outside [0, nslices)");
    if (a.ab_order < 1 || a.ab_order > 5) return qz_fail(QZ_EINVAL, "sweep: ab_order must be 1..5");
    if (a.nspecies < 0 || a.nspecies > QZ_MAX_SPECIES) return qz_fail(QZ_ERANGE, "sweep: at most 2 mobile species");
    if (a.ncf != (a.modes ? 18 : 6) || a.ncb != (a.modes ? 15 : 5) || a.ncd < (a.modes ? 9 : 3))
        return qz_fail(QZ_EINVAL, "sweep: component counts do not match modes");
    if (!a.ws || !a.fld || !a.diag || !a.bsrc || !a.bg || !a.lost) return qz_fail(QZ_EINVAL, "sweep: null array");
    if (a.groups < 0) return qz_fail(QZ_EINVAL, "sweep: negative groups");
    if (a.load)
        for (int s = 0; s < a.nspecies; ++s) {
            const qz_plasma_rings& rg = a.rings[s];
            if (rg.ppc < 1 || rg.ntheta < 1 || rg.nring < 0 || rg.nring > a.grid.N * rg.ppc || !rg.cs ||
                rg.nring * rg.ntheta != a.sp[s].np)
                return qz_fail(QZ_EINVAL, "sweep: the ring load of a species does not match its particle count");
        }
    if (a.groups > 1 && !a.mws) return qz_fail(QZ_EINVAL, "sweep: a run of several workgroups needs its workspace mws");
    if (a.traj && a.groups > 1) return qz_fail(QZ_EINVAL, "sweep: the trajectory buffer needs a one-workgroup run");
    for (int s = 0; s < a.nspecies; ++s)
        if (a.sp[s].np < 0 || a.sp[s].np > a.sp[s].cap || !a.sp[s].hist) return qz_fail(QZ_EINVAL, "sweep: bad species");
    return QZ_OK;
}

// The kernel reads its argument blocks from device memory for its whole duration.  They are staged in one
// buffer per (device, stream), reused only by later calls on the same stream, which the stream orders after
// the kernels that read it.  (A stream-ordered allocation per call could be handed to another stream while a
// kernel still reads it.)  The lock keeps the copy and the launch of one call together.
namespace {
struct ArgsBuf {
    qz_sweep_args* p = nullptr;
    int cap = 0;
    int* map = nullptr;         // block -> (run, group) of a multi-workgroup launch
    int mapcap = 0;
    std::vector<int> hmap;      // host side of the map (alive while the copy is staged)
};
std::mutex g_args_mu;
std::map<std::pair<int, hipStream_t>, ArgsBuf> g_args;
}  // namespace

static int sweep_many(const qz_sweep_args* runs, int n, void* stream) {
    if (!runs || n < 1) return qz_fail(QZ_EINVAL, "sweep: no runs");
    for (int i = 0; i < n; ++i) {
        const int rc = qz_validate_sweep(runs[i]);
        if (rc) return rc;
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    int dev = 0;
    QZ_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_args_mu);
    ArgsBuf& b = g_args[{dev, st}];
    if (b.cap < n) {   // grow: the old buffer may still be read by this stream's kernels
        if (b.p) {
            QZ_HIP(hipStreamSynchronize(st));
            QZ_HIP(hipFree(b.p));
            b.p = nullptr;
            b.cap = 0;
        }
        QZ_HIP(hipMalloc(reinterpret_cast<void**>(&b.p), sizeof(qz_sweep_args) * n));
        b.cap = n;
    }
    QZ_HIP(hipMemcpyAsync(b.p, runs, sizeof(qz_sweep_args) * n, hipMemcpyHostToDevice, st));
    bool multi = false;
    for (int i = 0; i < n; ++i) multi = multi || runs[i].groups > 1;
    if (!multi) return qz_sweep_launch(b.p, runs, n, st);
    // several workgroups per run: the block map, and every run's barrier counter and error flag at zero
    b.hmap = qz_sweep_block_map(runs, n);
    const int need = static_cast<int>(b.hmap.size());
    if (b.mapcap < need) {
        if (b.map) {
            QZ_HIP(hipStreamSynchronize(st));
            QZ_HIP(hipFree(b.map));
            b.map = nullptr;
            b.mapcap = 0;
        }
        QZ_HIP(hipMalloc(reinterpret_cast<void**>(&b.map), sizeof(int) * need));
        b.mapcap = need;
    }
    QZ_HIP(hipMemcpyAsync(b.map, b.hmap.data(), sizeof(int) * need, hipMemcpyHostToDevice, st));
    for (int i = 0; i < n; ++i) {
        if (!runs[i].mws) return qz_fail(QZ_EINVAL, "sweep: in a multi-workgroup launch every run needs mws");
        const int rc = qz_zero_async(runs[i].mws, 64 * sizeof(double), st);
        if (rc) return rc;
    }
    return qz_sweep_multi_launch(b.p, b.map, runs, n, st);
}

extern "C" int qz_sweep(const qz_sweep_args* args, void* stream) { return sweep_many(args, 1, stream); }
extern "C" int qz_sweep_release(void* stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    int dev = 0;
    QZ_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_args_mu);
    auto it = g_args.find({dev, st});
    if (it == g_args.end()) return QZ_OK;
    QZ_HIP(hipStreamSynchronize(st));   // its kernels may still read the block
    if (it->second.p) QZ_HIP(hipFree(it->second.p));
    if (it->second.map) QZ_HIP(hipFree(it->second.map));
    g_args.erase(it);
    return QZ_OK;
}
extern "C" int qz_sweep_batched(const qz_sweep_args* runs, int nruns, void* stream) {
    return sweep_many(runs, nruns, stream);
}

// ---------------------------------------------------------------------------- the sweep without allocation
// For callers that cannot allocate device memory (code under HIP graph capture, serving loops): one run's sweep
// whose argument block and workspace live in this library's static device array `scratch`, so the call makes
// no allocation at all.  Every GPU holds its own copy of the array for the life of the process; its address on
// a device is looked up once, with that device current (hipGetSymbolAddress), and only that address is handed
// to kernels and copies.  Calls on one GPU share the array: two calls whose sweeps overlap in time race, and
// the workspace keeps what the last call left (a slice range continuing an earlier one reads its B+ from it).
namespace {
constexpr size_t kScratchArgBytes = 4096;                       // one qz_sweep_args block, rounded up
constexpr int kScratchMaxM = QZ_NOALLOC_MAX_NODES;              // grid nodes N + 1
constexpr size_t kScratchBytes = kScratchArgBytes + sizeof(double) * QZ_SWEEP_WS_ARRAYS * kScratchMaxM;
static_assert(sizeof(qz_sweep_args) <= kScratchArgBytes, "the argument block must fit its scratch slot");
}  // namespace

__device__ __align__(256) char scratch[kScratchBytes];

namespace {
std::mutex g_scratch_mu;
std::map<int, char*> g_scratch_ptr;   // device -> address of `scratch` on it

int scratch_on_current_device(char** out) {
    int dev = 0;
    QZ_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    auto it = g_scratch_ptr.find(dev);
    if (it == g_scratch_ptr.end()) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return qz_fail_hip(e, "qz_sweep_noalloc: hipGetSymbolAddress(scratch)");
        it = g_scratch_ptr.emplace(dev, static_cast<char*>(p)).first;
    }
    *out = it->second;
    return QZ_OK;
}
}  // namespace

namespace qz {
// the argument block goes to device memory as a kernel argument: a graph that captures the call keeps the values
// in its kernel node (a copy from host memory would read the caller's memory again at every replay)
__global__ void put_args_kernel(qz_sweep_args a, qz_sweep_args* __restrict__ dst) {
    constexpr int nw = static_cast<int>(sizeof(qz_sweep_args) / sizeof(unsigned int));
    const unsigned int* src = reinterpret_cast<const unsigned int*>(&a);
    unsigned int* out = reinterpret_cast<unsigned int*>(dst);
    for (int i = threadIdx.x; i < nw; i += blockDim.x) out[i] = src[i];
}
}  // namespace qz

extern "C" int qz_sweep_noalloc(const qz_sweep_args* args, void* stream) {
    if (!args) return qz_fail(QZ_EINVAL, "qz_sweep_noalloc: null argument");
    const int M = args->grid.N + 1;
    if (M > kScratchMaxM)
        return qz_fail(QZ_ERANGE, "qz_sweep_noalloc: " + std::to_string(M) + " grid nodes exceed the scratch array's " +
                                      std::to_string(kScratchMaxM));
    char* base = nullptr;
    const int rc = scratch_on_current_device(&base);
    if (rc) return rc;
    if (args->groups > 1) return qz_fail(QZ_EINVAL, "qz_sweep_noalloc: one workgroup per run (groups 0 or 1)");
    qz_sweep_args a = *args;
    a.ws = reinterpret_cast<double*>(base + kScratchArgBytes);   // the run's workspace: the scratch after the block
    const int v = qz_validate_sweep(a);
    if (v) return v;
    hipStream_t st = static_cast<hipStream_t>(stream);
    qz_sweep_args* dev_args = reinterpret_cast<qz_sweep_args*>(base);
    static_assert(sizeof(qz_sweep_args) % sizeof(unsigned int) == 0, "the block is copied in 4-byte words");
    hipLaunchKernelGGL(qz::put_args_kernel, dim3(1), dim3(64), 0, st, a, dev_args);
    QZ_HIP(hipGetLastError());
    return qz_sweep_launch(dev_args, &a, 1, st);
}
