// Host runtime of the Fock-build engine (native C ABI, include/quickfock.h).
//
// Replaces QUICK's GPU host side for the two-electron path:
//   gpu_upload_basis_ Q-shell split and sort   (src/gpu/hip/gpu.cu:1782-2134)
//   gpu_upload_cutoff_matrix_ pair-list build  (src/gpu/hip/gpu.cu:879-1484)
//   get2e launches                             (src/gpu/hip/gpu_get2e.cu:595-638)
//   download / symmetrise / accumulate         (src/gpu/gpu_get2e_getxc_drivers.h:27-121)
// but keeps everything device-resident: pair data and task lists are built
// once per geometry (O(n log n) sorts), a build only uploads nothing, screens
// the density on the device, launches one kernel per class and symmetrises.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <mutex>
#include <map>
#include <memory>
#include <numeric>
#include <string>
#include <vector>

#include "../../include/quickfock.h"
#include "gen/grad_launchers.h"
#include "gen/launchers.h"
#include "qf_types.h"

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg)
{
    // a failed HIP call is reported here: the next call of this library, which asks
    // for the runtime's last error, is not to report it again
    if (code == QF_ERR_HIP || code == QF_ERR_MEMORY) (void)hipGetLastError();
    g_err = msg;
    return code;
}

#define QF_HIP(call)                                                                              \
    do {                                                                                          \
        hipError_t _e = (call);                                                                   \
        if (_e != hipSuccess)                                                                     \
            return fail(QF_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(_e));         \
    } while (0)

constexpr double kPi = 3.14159265358979323846264338327950288;
const double kX0 = 2.0 * std::pow(kPi, 2.5);   // QUICK's X0 (quick_constants_module.f90:61)

inline int pair_class(int La, int Lb) { return La * (La + 1) / 2 + Lb; }
const char* const kDirectFp32Refused =
    "the direct-atomic kernels run FP64 only (their FP32 form gave wrong Fock matrices on gfx950 and is not "
    "built); FP32 halves run on the LDS-tile kernel";
constexpr int kCoopWindow = 2;   // kets per task of the wave-per-quartet kernels
constexpr int kNPC = 10;   // pair classes (La >= Lb) for s, p, d, f
constexpr size_t kMaxTileLds = 64 * 1024;   // dynamic LDS of one tile workgroup
const int kClassL[kNPC][2] = {{0, 0}, {1, 0}, {1, 1}, {2, 0}, {2, 1}, {2, 2}, {3, 0}, {3, 1}, {3, 2}, {3, 3}};
inline int ncart(int L) { return (L + 1) * (L + 2) / 2; }

template <typename T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
    ~DevBuf() { release(); }
    void release()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    hipError_t resize(size_t count)
    {
        if (count <= n && p) return hipSuccess;
        release();
        if (count == 0) return hipSuccess;
        hipError_t e = hipMalloc(&p, count * sizeof(T));
        if (e == hipSuccess) n = count;
        return e;
    }
    hipError_t upload(const std::vector<T>& v)
    {
        hipError_t e = resize(v.size());
        if (e != hipSuccess || v.empty()) return e;
        return hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice);
    }
    size_t bytes() const { return n * sizeof(T); }
};

struct QShell {
    int L, atom, shell, fn, nprim, pstart, qfin;
};

struct HostBlock {
    int cls = 0, K = 0;
    std::vector<qf::PairInfo> info;
    std::vector<int> bperm;                      // pair indices grouped by first Q-shell
    std::vector<std::pair<int, int>> groups;     // [start, end) in bperm, one per first Q-shell
    std::vector<double> prim;   // PF_N * K * n, filled at finalisation
    std::vector<std::vector<double>> rows;   // per pair: PF_N*K values (field-major)
    std::vector<int> colf;                   // compact column -> basis function
};

// --------------------------------------------------------------------------
// Side streams.  The class launches of a build are independent (they only
// add into G with atomics), and most of them cannot fill the GPU: a launch
// of a small molecule is one wave's latency long, a launch of a large one
// ends in a tail of few waves.  A build therefore forks from the caller's
// stream onto kSide more streams of default priority and joins them again
// before G is summed, all by events, so the caller's stream order (and a
// capture of it) covers everything.  Four streams in all, the hardware
// queues a process has.  One stream -> four, ms per build: water 6-31G*
// (host call) 0.35 -> 0.21, glycine 6-31G** 1.51 -> 0.95, (H2O)8 cc-pVDZ
// 2.73 -> 1.48, ethane def2-TZVP 4.47 -> 2.79, (H2O)8+ open shell 3.71 ->
// 1.54, (H2O)32 6-31G* 13.9 -> 11.6, (Gly)10 mixed 33.4 -> 30.7.
//
// A set belongs to one engine or batch while that lives (a set that takes
// part in a capture cannot serve another thread's builds); at most kKeep
// sets per device are kept when their owners have gone.
// --------------------------------------------------------------------------
constexpr int kSide = 3;

struct SideStreams {
    int device = -1;
    hipStream_t s[kSide] = {};
    hipEvent_t fork = nullptr, done[kSide] = {};

    bool create(int dev)
    {
        device = dev;
        bool ok = hipEventCreateWithFlags(&fork, hipEventDisableTiming) == hipSuccess;
        for (int k = 0; ok && k < kSide; ++k)
            ok = hipStreamCreateWithFlags(&s[k], hipStreamNonBlocking) == hipSuccess &&
                 hipEventCreateWithFlags(&done[k], hipEventDisableTiming) == hipSuccess;
        return ok;
    }
    ~SideStreams()
    {
        if (fork) (void)hipEventDestroy(fork);
        for (int k = 0; k < kSide; ++k) {
            if (s[k]) (void)hipStreamDestroy(s[k]);
            if (done[k]) (void)hipEventDestroy(done[k]);
        }
    }
};

class SidePool {
public:
    static SidePool& get()
    {
        // never destroyed: the streams it keeps must not outlive the HIP runtime
        static SidePool* pool = new SidePool();
        return *pool;
    }
    SideStreams* take(int device)
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            for (size_t k = 0; k < free_.size(); ++k)
                if (free_[k]->device == device) {
                    SideStreams* ss = free_[k];
                    free_.erase(free_.begin() + k);
                    return ss;
                }
        }
        SideStreams* ss = new SideStreams();
        if (ss->create(device)) return ss;
        (void)hipGetLastError();   // not an error of the build, which ends by asking for the last one
        delete ss;
        return nullptr;            // the caller runs on its own stream alone
    }
    void give(SideStreams* ss)
    {
        if (!ss) return;
        {
            std::lock_guard<std::mutex> lk(mu_);
            int same = 0;
            for (auto* x : free_) same += x->device == ss->device;
            if (same < kKeep) {
                free_.push_back(ss);
                return;
            }
        }
        delete ss;
    }

private:
    static constexpr int kKeep = 8;
    std::mutex mu_;
    std::vector<SideStreams*> free_;
};

bool is_capturing(hipStream_t s)
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) {
        (void)hipGetLastError();
        return true;    // unknown: only plain launches
    }
    return st != hipStreamCaptureStatusNone;
}

// Id of the capture that s takes part in, 0 for none.
unsigned long long capture_of(hipStream_t s)
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (hipStreamGetCaptureInfo(s, &st, &id) != hipSuccess) {
        (void)hipGetLastError();
        return ~0ull;
    }
    return st == hipStreamCaptureStatusNone ? 0 : id;
}

// Whether work on s may be forked onto the side streams: those that took part in a
// capture belong to it until it ends, and can serve no other stream.
bool side_free(const SideStreams& side, hipStream_t s)
{
    const unsigned long long of = capture_of(s);
    for (hipStream_t q : side.s) {
        const unsigned long long id = capture_of(q);
        if (id != 0 && id != of) return false;
    }
    return true;
}

// Makes sure `side` has its streams, unless s is being captured (creating
// streams is no work for a capture; without them everything runs on s).
bool side_ready(SideStreams*& side, int device, hipStream_t s)
{
    if (side) return true;
    if (is_capturing(s)) return false;
    side = SidePool::get().take(device);
    return side != nullptr;
}

// --------------------------------------------------------------------------
// Device helper kernels
// --------------------------------------------------------------------------
// Opening kernel of a build, in one launch: the descriptors the class kernels
// read (from the kernel arguments, so a captured build keeps its own), zeroed
// G accumulators, the density screen matrix and, for an open-shell build, the
// total and spin densities.  Before, two copies and up to four kernels.
//
// Screen matrix: QUICK's cshell_density_cutoff (cutoff.fh:65-92), max |P_ij|
// over the functions of the two original shells, or, with Pb,
// oshell_density_cutoff (cutoff.fh:16-89), max of max(|Pa+Pb|, |Pa|, |Pb|).
struct OpenArgs {
    qf::MolDesc md, mx;              // descriptors, written to *dmd and *dmx where not null
    qf::MolDesc *dmd, *dmx;
    const double *Pa, *Pb;           // densities (Pb null: closed shell)
    double *Pc, *Pd;                 // where not null: the densities are in host memory, their copies on the device
    double *Pt, *Ps;                 // open shell: Pa + Pb and Pa - Pb
    double *G, *G2;                  // ng doubles each to zero (null: none)
    size_t ng;
    double* cm;                      // screen matrix to compute (null: the caller's is used)
    const int *f0, *f1;              // first and last function of every shell
    int n, nshell;
};

__global__ __launch_bounds__(256) void k_open(const OpenArgs a)
{
    const size_t first = blockIdx.x * (size_t)blockDim.x + threadIdx.x, step = (size_t)gridDim.x * blockDim.x;
    if (first == 0) {
        if (a.dmd) *a.dmd = a.md;
        if (a.dmx) *a.dmx = a.mx;
    }
    if (a.Pc) {
        // a workgroup per shell: its rows come over the bus once, one contiguous read
        for (int I = blockIdx.x; I < a.nshell; I += gridDim.x) {
            const size_t r0 = (size_t)a.f0[I] * a.n, r1 = (size_t)(a.f1[I] + 1) * a.n;
            for (size_t idx = r0 + threadIdx.x; idx < r1; idx += blockDim.x) {
                const double p = a.Pa[idx];
                a.Pc[idx] = p;
                if (a.Pb) {
                    const double q = a.Pb[idx];
                    a.Pd[idx] = q;
                    a.Pt[idx] = p + q;
                    a.Ps[idx] = p - q;
                }
            }
            __syncthreads();
            if (a.cm)
                for (int J = threadIdx.x; J < a.nshell; J += blockDim.x) {
                    double m = 0.0;
                    for (int i = a.f0[I]; i <= a.f1[I]; ++i)
                        for (int j = a.f0[J]; j <= a.f1[J]; ++j) {
                            const double p = a.Pc[(size_t)i * a.n + j], q = a.Pb ? a.Pd[(size_t)i * a.n + j] : 0.0;
                            m = fmax(m, fmax(fabs(p + q), fmax(fabs(p), fabs(q))));
                        }
                    a.cm[(size_t)I * a.nshell + J] = m;
                }
        }
    } else if (a.cm) {
        for (size_t idx = first; idx < (size_t)a.nshell * a.nshell; idx += step) {
            const int I = (int)(idx / a.nshell), J = (int)(idx % a.nshell);
            double m = 0.0;
            for (int i = a.f0[I]; i <= a.f1[I]; ++i)
                for (int j = a.f0[J]; j <= a.f1[J]; ++j) {
                    const double p = a.Pa[(size_t)i * a.n + j], q = a.Pb ? a.Pb[(size_t)i * a.n + j] : 0.0;
                    m = fmax(m, fmax(fabs(p + q), fmax(fabs(p), fabs(q))));
                }
            a.cm[idx] = m;
        }
    }
    if (a.Pt && !a.Pc)
        for (size_t idx = first; idx < (size_t)a.n * a.n; idx += step) {
            const double p = a.Pa[idx], q = a.Pb[idx];
            a.Pt[idx] = p + q;
            a.Ps[idx] = p - q;
        }
    if (a.G)
        for (size_t i = first; i < a.ng; i += step) a.G[i] = 0.0;
    if (a.G2)
        for (size_t i = first; i < a.ng; i += step) a.G2[i] = 0.0;
}

void open_build(const OpenArgs& a, qf::LaunchTo& q)
{
    const size_t work = std::max({(size_t)a.n * a.n, a.G ? a.ng : (size_t)0, a.Pc ? (size_t)a.nshell * 256 : (size_t)0});
    const int grid = (int)std::min<size_t>(2048, (work + 255) / 256);
    q(k_open, dim3(grid), dim3(256), 0, a);
}

__global__ void k_zero(double* __restrict__ p, size_t count)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0.0;
}

// Closing kernel of a build.  Closed shell: G = sum over copies of (Gt +
// Gt^T), F += G.  Open shell (Gt2): A = the sum of Gt (J and exchange of Pt), B
// = the sum of Gt2 (exchange of Ps); Fa += A + B, Fb += A - B, Gs = A.
struct CloseArgs {
    const double *Gt, *Gt2;
    double *Gs, *F, *F2;
    double *H, *H2;          // in host memory: what F and F2 would have added (null: none)
    int replicas, n;
};

__global__ __launch_bounds__(256) void k_close(const CloseArgs a)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= a.n * a.n) return;
    const int i = idx / a.n, j = idx % a.n;
    const size_t n2 = (size_t)a.n * a.n, ij = (size_t)i * a.n + j, ji = (size_t)j * a.n + i;
    double g = 0.0, h = 0.0;
    for (int r = 0; r < a.replicas; ++r) g += a.Gt[r * n2 + ij] + a.Gt[r * n2 + ji];
    if (a.Gt2)
        for (int r = 0; r < a.replicas; ++r) h += a.Gt2[r * n2 + ij] + a.Gt2[r * n2 + ji];
    a.Gs[idx] = g;
    if (a.F) a.F[idx] += g + h;
    if (a.F2) a.F2[idx] += g - h;
    if (a.H) a.H[idx] = g + h;
    if (a.H2) a.H2[idx] = g - h;
}

void close_build(const CloseArgs& a, qf::LaunchTo& q)
{
    q(k_close, dim3((a.n * a.n + 255) / 256), dim3(256), 0, a);
}

__global__ void k_copy(const double* __restrict__ from, double* __restrict__ to, int count)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) to[i] = from[i];
}

// Pinned host memory through which calls with host matrices pass them: the
// opening kernel reads the densities from it and the closing kernel writes the
// result to it.  Before, every matrix had a copy of its own that waited for the
// GPU.  Host to host, us, copies -> pinned memory: water 6-31G* (19 functions) Fock
// 107 -> 86, open shell 184 -> 101, gradient 159 -> 138; ethane 6-31G* (42) 182 -> 166,
// 310 -> 238, 326 -> 304; glycine 6-31G** (100) 441 -> 418, 589 -> 539, 1522 -> 1504;
// (H2O)8 cc-pVDZ (200) Fock 1028 -> 1008, gradient 2118 -> 2104.  The gain, 15-20 us a
// matrix, is within 2 % from 200 functions (80000 doubles) on, where the copies stay.
// A call takes a buffer, waits for the GPU and gives it back; at most kKeep
// wait in the pool, shared by all threads and devices.
constexpr size_t kStageDoubles = 80000;
class StagePool {
public:
    static StagePool& get()
    {
        static StagePool* pool = new StagePool;   // never destroyed: engines may outlive static objects
        return *pool;
    }
    double* take()
    {
        {
            std::lock_guard<std::mutex> lock(mu_);
            if (!free_.empty()) {
                double* p = free_.back();
                free_.pop_back();
                return p;
            }
        }
        void* p = nullptr;
        if (hipHostMalloc(&p, kStageDoubles * sizeof(double), hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        return (double*)p;
    }
    void give(double* p)
    {
        {
            std::lock_guard<std::mutex> lock(mu_);
            if (free_.size() < kKeep) {
                free_.push_back(p);
                return;
            }
        }
        (void)hipHostFree(p);
    }

private:
    static constexpr size_t kKeep = 8;
    std::mutex mu_;
    std::vector<double*> free_;
};

// A buffer for `count` doubles, or none (p null) where that is too many; waits
// for the null stream before it goes back.
struct Stage {
    double* p;
    explicit Stage(size_t count) : p(count <= kStageDoubles ? StagePool::get().take() : nullptr) {}
    ~Stage()
    {
        if (!p) return;
        if (!done) (void)hipStreamSynchronize(nullptr);
        StagePool::get().give(p);
    }
    int wait()
    {
        QF_HIP(hipStreamSynchronize(nullptr));
        done = true;
        return QF_OK;
    }
    bool done = false;
};

// The launches of one kind of build as an instantiated graph.
struct Replay {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hipGraphNode_t first = nullptr, last = nullptr;   // the opening and the closing kernel
    OpenArgs open{};        // arguments that `first` and `last` hold
    CloseArgs close{};
    int uses = 0;           // builds of this kind since the last prepare
    bool failed = false;    // could not be built: the launches stay eager
    std::vector<std::pair<hipGraph_t, hipGraphExec_t>> old;   // put aside, may still run
    // Puts the graph aside without a wait: a setter may be called while a stream is
    // captured, and a wait would end the capture.  Bounded: builds outside a capture
    // give what was put aside back (sweep).
    void retire()
    {
        if (old.size() >= 16) sweep();
        if (exec)
            old.push_back({graph, exec});
        else if (graph)
            (void)hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
        uses = 0;
        failed = false;
    }
    void sweep()
    {
        if (old.empty()) return;
        (void)hipDeviceSynchronize();   // they may still run
        for (auto& x : old) {
            (void)hipGraphExecDestroy(x.second);
            (void)hipGraphDestroy(x.first);
        }
        old.clear();
        (void)hipGetLastError();
    }
    void drop()
    {
        retire();
        sweep();
    }
};

// Counts, per quartet class, the quartets and primitive quartets that pass
// the screens (same tests as the Fock kernel); used for the FLOP model.
// grad = 1: the gradient's screen (md.cutoff is gradCutoff, quartets on one
// atom skipped).
__global__ void k_count(const qf::Task* __restrict__ tasks, int ntasks, const qf::PairBlock* __restrict__ blocks,
                        const qf::MolDesc* __restrict__ mols, unsigned long long* __restrict__ counts, int slot,
                        int fp32, int grad)
{
    const int tix = blockIdx.x;
    if (tix >= ntasks) return;
    const qf::Task t = tasks[tix];
    const qf::PairBlock bb = blocks[t.bra_block];
    const qf::PairBlock kb = blocks[t.ket_block];
    const qf::MolDesc md = mols[bb.mol];
    const int lane = threadIdx.x;
    if (lane >= t.ket_count) return;
    const int j = t.ket_start + lane;
    const qf::PairInfo ki = kb.info[j];
    const int ns = md.nshell;
    const double* cm = md.cutmat;
    unsigned long long nq = 0, np = 0;
    for (int kk = t.kb; kk < t.ke; ++kk) {
        const int i = bb.bperm[kk];
        const qf::PairInfo bi = bb.info[i];
        double dn = 4.0 * cm[bi.sa * ns + bi.sb];
        dn = fmax(dn, 4.0 * cm[ki.sa * ns + ki.sb]);
        dn = fmax(dn, cm[bi.sa * ns + ki.sb]);
        dn = fmax(dn, cm[bi.sa * ns + ki.sa]);
        dn = fmax(dn, cm[bi.sb * ns + ki.sa]);
        dn = fmax(dn, cm[bi.sb * ns + ki.sb]);
        const double y = bi.ycut * ki.ycut;
        if (!(y > md.cutoff && y * dn > md.cutoff)) continue;
        if (t.same_block && j > i) continue;
        if (fp32 ? !(y < md.split) : !(t.all_fp64 || y >= md.split)) continue;
        if (grad) {
            const int a = md.shell_atom[bi.sa];
            if (a == md.shell_atom[bi.sb] && a == md.shell_atom[ki.sa] && a == md.shell_atom[ki.sb]) continue;
        }
        if (t.pb == 0 && t.qb == 0) ++nq;   // a quartet spread over several tasks counts once
        for (int ip = t.pb; ip < t.pe; ++ip) {
            const double c1 = dn * bb.prim[(qf::PF_CUT * bb.K + ip) * bb.n + i];
            for (int jp = t.qb; jp < t.qe; ++jp)
                if (c1 * kb.prim[(qf::PF_CUT * kb.K + jp) * kb.n + j] > md.primlim) ++np;
        }
    }
    atomicAdd(&counts[2 * slot], nq);
    atomicAdd(&counts[2 * slot + 1], np);
}

}  // namespace

// ==========================================================================
struct qf_engine {
    int device = 0;
    // molecule + basis (host)
    int natom = 0;
    std::vector<double> xyz;
    int nshell = 0, nprim = 0, nbasis = 0;
    std::vector<int> s_atom, s_lmin, s_lmax, s_nprim, s_pstart, s_fstart;
    std::vector<double> exps, coef;
    std::vector<QShell> qs;
    // screening
    std::vector<double> ycut, cutprim;
    bool have_schwarz = false;
    double cutoff = 1e-12, primlim = 1e-13, hyb = 1.0;
    double grad_cutoff = -1.0;   // QUICK's gradCutoff (qf_set_grad_cutoff); <= 0: the integral cutoff
    bool grad_lane = true;       // per-lane gradient kernels where a class has one (qf_set_grad_kernel)
    // pair lists and task windows cover every quartet either screen can keep
    double list_cutoff() const { return grad_cutoff > 0.0 ? std::min(cutoff, grad_cutoff) : cutoff; }
    int prec = QF_PREC_FP64;
    double split = 1e-4;
    int split_lmin = -1;     // classes with La+Lb+Lc+Ld >= split_lmin are split in mixed builds (-1: by size)
    double split_thr = 0.0;  // Ycut_ij*Ycut_kl below which quartets run in FP32
    int replicas = 8;        // copies of G the atomics are spread over
    int shuffle = 1;         // permute tasks inside a launch (decorrelates atomic targets)
    int tile = 1;            // accumulate exchange terms in LDS tiles (fock_tile_kernel)
    int tile_waves = 4;      // max waves per tile workgroup
    int tile_tasks = 0;      // max tasks per tile workgroup (0: 1 or 2 up to 256 functions, 4 up to 400, 16 above)
    int lds_budget = 64 * 1024;
    int persist = 0;         // grid cap of the class launches (0: one workgroup per task / group)
    int prim_piece = 0;      // primitive pairs per task piece: 0 auto, < 0 never split
    struct ClassTune {
        int tile = -1, waves = 0, tpg = 0, mmax = 0;   // <0 / 0: engine default
        int piece = 0;                                  // primitive pairs per piece: 0 engine default, < 0 none
        int os = -1;   // open-shell form: -1 default (2), 0 fused, 1 two passes, 2 fused lean (tile kernels)
        int grad = -1; // gradient kernel: -1 engine default, 0 wave-per-quartet, 1 per-lane
        int split = -1; // mixed builds: -1 engine rule (split_lmin), 0 all FP64, 1 split
    };
    ClassTune ctune[kNPC][kNPC];
    // pair blocks
    std::vector<HostBlock> blocks;
    std::vector<qf::PairBlock> hblocks;
    std::vector<qf::Task> tasks;
    std::vector<qf::TileGroup> groups;
    struct Launch {
        int cb, ck, fp32, offset, count;
        int tile, goffset, gcount, waves;
        size_t lds;
        size_t lds_os;   // open-shell pass with a second exchange tile (0: it does not fit)
        int os_split;    // open-shell builds run this class as two closed-shell passes
        int os_lean;     // ... or, on the tile kernel, in the fused lean form
        int closed_only;             // the tile kernel has no open-shell and no gradient form: these run the
        int alt_offset, alt_count;   // class on the wave-per-quartet kernels, with tasks of their own in d_alt
        size_t gslot;    // first double of its region of the global slot buffer (classes that need one)
    };
    std::vector<Launch> launches;
    struct Fused {           // classes of `launches` that share a launch
        int kernel;          // qf::fuse_kernel
        int offset, count;   // its workgroups in d_fused
        int waves;
        size_t lds, gslot;
        double seconds;      // estimate
    };
    std::vector<Fused> fused;
    struct Plan {
        std::vector<std::pair<int, int>> order;   // (launch index, or ~ the index into fused; stream 0..kSide)
        double gain = 0.0;                        // seconds the forked order saves (estimate)
    };
    Plan plan[4];                             // closed shell, open shell, gradient; one launch per class
    bool shared = false;                      // up to the sizes of shares_launches
    size_t grad_slots = 0;                    // doubles of global slots that the gradient's shared launches need
    SideStreams* side = nullptr;              // taken at the first forked build
    Replay replay[3];                         // closed shell, open shell, gradient
    void drop_replays()
    {
        for (auto& r : replay) r.drop();
    }
    bool prepared = false;
    unsigned long long generation = 0;   // bumped by every prepare(): batches check it
    bool built = false;                  // a build has run since the last prepare()
    bool count_cm_own = false;           // ... and screened with the engine's own Cutmatrix (d_cm)
    qf_stats stats{};
    double flops_last = -1.0;
    // device
    DevBuf<qf::PairInfo> d_info;
    DevBuf<double> d_prim;
    DevBuf<int> d_perm;
    DevBuf<qf::PairBlock> d_blocks;
    DevBuf<qf::MolDesc> d_mol;
    DevBuf<qf::Task> d_tasks;
    DevBuf<qf::Task> d_alt;
    DevBuf<qf::TileGroup> d_groups;
    DevBuf<qf::FusedBlock> d_fused;
    DevBuf<int> d_colf;
    DevBuf<double> d_Gt, d_Gs, d_cm, d_P;
    DevBuf<double> d_Pb, d_Pt, d_Ps, d_Fa, d_Fb;   // open-shell builds (allocated on first use)
    DevBuf<double> d_Gt2;                           // their second exchange accumulators (replicas x n^2)
    DevBuf<double> d_zero;                          // nbasis^2 zeros: Coulomb density of an exchange-only pass
    DevBuf<int> d_shells;        // per shell: first and last function, atom (nshell each)
    const int* shell_f0() const { return d_shells.p; }
    const int* shell_f1() const { return d_shells.p + nshell; }
    const int* shell_at() const { return d_shells.p + 2 * nshell; }
    DevBuf<unsigned long long> d_counts;
    DevBuf<double> d_cscratch;   // global slots of the wave-per-quartet classes that need them
    DevBuf<double> d_gscratch;   // global slots of the gradient classes that need them (on first use)
    DevBuf<double> d_grad;       // gradient of the host entry point (on first use)
    bool grad_built = false;     // a gradient has run since the last prepare() (counts need it) ...
    bool grad_cm_own = false;    // ... screened with the engine's own Cutmatrix
    // per-launch timing (HIP events on the build stream)
    bool timing = false;
    std::vector<hipEvent_t> ev_pool;
    size_t ev_used = 0;
    std::vector<int> ev_launch;        // launch index of each recorded (start, stop) pair
    ~qf_engine()
    {
        drop_replays();
        for (hipEvent_t ev : ev_pool) (void)hipEventDestroy(ev);
        SidePool::get().give(side);
    }

    int set_device() { return hipSetDevice(device) == hipSuccess ? QF_OK : fail(QF_ERR_BADDEVICE, "hipSetDevice"); }
};

namespace {

// Q-shells: an SP shell becomes an s and a p Q-shell (gpu.cu:1884-1887).
void build_qshells(qf_engine* e)
{
    e->qs.clear();
    for (int s = 0; s < e->nshell; ++s) {
        int off = 0;
        for (int L = e->s_lmin[s]; L <= e->s_lmax[s]; ++L) {
            e->qs.push_back({L, e->s_atom[s], s, e->s_fstart[s] + off, e->s_nprim[s], e->s_pstart[s], e->s_lmax[s]});
            off += ncart(L);
        }
    }
}

double cutprim_sym(const qf_engine* e, int pa, int pb)
{
    // QUICK fills cutprim for shell order II <= JJ only; the value is
    // symmetric, so take whichever triangle holds it.
    const size_t jb = e->nprim;
    return std::max(e->cutprim[pa * jb + pb], e->cutprim[pb * jb + pa]);
}

// One canonical pair (La >= Lb; equal L: qa >= qb).  If ip >= 0 the pair
// holds the single primitive pair (ip, jp) (cutprim evaluation).
void make_pair(const qf_engine* e, int qa, int qb, int ip, int jp, bool use_cut, qf::PairInfo& info,
               std::vector<double>& row, int& K)
{
    const QShell& a = e->qs[qa];
    const QShell& b = e->qs[qb];
    const double* A = &e->xyz[3 * a.atom];
    const double* B = &e->xyz[3 * b.atom];
    info.qa = qa;
    info.qb = qb;
    info.fa = a.fn;
    info.fb = b.fn;
    info.sa = a.shell;
    info.sb = b.shell;
    info.qfs = a.qfin + e->s_lmax[b.shell];
    info.id = 0;
    info.ycut = e->have_schwarz ? e->ycut[(size_t)a.shell * e->nshell + b.shell] : 1.0;
    double AB2 = 0.0;
    for (int d = 0; d < 3; ++d) {
        info.A[d] = A[d];
        info.AB[d] = A[d] - B[d];
        AB2 += info.AB[d] * info.AB[d];
    }
    info.cola = info.colb = 0;
    struct Prim {
        double v[qf::PF_N];
    };
    std::vector<Prim> prims;
    const double sx0 = std::sqrt(kX0);
    for (int i = 0; i < a.nprim; ++i)
        for (int j = 0; j < b.nprim; ++j) {
            if (ip >= 0 && (i != ip || j != jp)) continue;
            const int pa = a.pstart + i, pb = b.pstart + j;
            const double al = e->exps[pa], be = e->exps[pb];
            const double z = al + be;
            Prim p;
            p.v[qf::PF_ZETA] = z;
            p.v[qf::PF_OOZ2] = 0.5 / z;
            for (int d = 0; d < 3; ++d) p.v[qf::PF_PX + d] = (A[d] * al + B[d] * be) / z;
            // Kpri * c_a * c_b (eri.fh:120-140) with sqrt(X0) per pair, so a
            // quartet carries X0 once (eri.fh:514).
            const double kpri = std::exp(-al * be / z * AB2) / z;
            p.v[qf::PF_KC] = sx0 * kpri * e->coef[(size_t)pa * 4 + a.L] * e->coef[(size_t)pb * 4 + b.L];
            p.v[qf::PF_CUT] = use_cut ? cutprim_sym(e, pa, pb) : 1.0;
            p.v[qf::PF_ALPHA] = al;
            prims.push_back(p);
        }
    std::stable_sort(prims.begin(), prims.end(),
                     [](const Prim& x, const Prim& y) { return x.v[qf::PF_CUT] > y.v[qf::PF_CUT]; });
    K = (int)prims.size();
    row.assign((size_t)qf::PF_N * K, 0.0);
    for (int f = 0; f < qf::PF_N; ++f)
        for (int k = 0; k < K; ++k) row[(size_t)f * K + k] = prims[k].v[f];
}

// Assemble host blocks into flat device arrays; fills hblocks (device pointers).
int upload_blocks(qf_engine* e, std::vector<HostBlock>& blocks, DevBuf<qf::PairInfo>& d_info,
                  DevBuf<double>& d_prim, std::vector<qf::PairBlock>& out, int mol, DevBuf<int>* d_perm = nullptr,
                  DevBuf<int>* d_colf = nullptr)
{
    size_t ninfo = 0, nprimv = 0;
    for (auto& b : blocks) {
        ninfo += b.info.size();
        nprimv += (size_t)qf::PF_N * b.K * b.info.size();
    }
    std::vector<qf::PairInfo> info;
    info.reserve(ninfo);
    std::vector<double> prim(nprimv);
    std::vector<size_t> ioff, poff;
    size_t po = 0;
    for (auto& b : blocks) {
        ioff.push_back(info.size());
        poff.push_back(po);
        const size_t n = b.info.size();
        info.insert(info.end(), b.info.begin(), b.info.end());
        for (size_t j = 0; j < n; ++j)
            for (int f = 0; f < qf::PF_N; ++f)
                for (int k = 0; k < b.K; ++k) prim[po + ((size_t)f * b.K + k) * n + j] = b.rows[j][(size_t)f * b.K + k];
        po += (size_t)qf::PF_N * b.K * n;
    }
    QF_HIP(d_info.upload(info));
    QF_HIP(d_prim.upload(prim));
    std::vector<int> perm;
    std::vector<size_t> permoff;
    for (auto& b : blocks) {
        permoff.push_back(perm.size());
        perm.insert(perm.end(), b.bperm.begin(), b.bperm.end());
    }
    if (d_perm) QF_HIP(d_perm->upload(perm));
    std::vector<int> colf;
    std::vector<size_t> coloff;
    for (auto& b : blocks) {
        coloff.push_back(colf.size());
        colf.insert(colf.end(), b.colf.begin(), b.colf.end());
    }
    if (d_colf) QF_HIP(d_colf->upload(colf));
    out.clear();
    for (size_t k = 0; k < blocks.size(); ++k) {
        qf::PairBlock pb;
        pb.info = d_info.p + ioff[k];
        pb.prim = d_prim.p + poff[k];
        pb.bperm = (d_perm && !blocks[k].bperm.empty()) ? d_perm->p + permoff[k] : nullptr;
        pb.colf = (d_colf && !blocks[k].colf.empty()) ? d_colf->p + coloff[k] : nullptr;
        pb.ncol = (int)blocks[k].colf.size();
        pb.pad = 0;
        pb.n = (int)blocks[k].info.size();
        pb.K = blocks[k].K;
        pb.cls = blocks[k].cls;
        pb.mol = mol;
        out.push_back(pb);
    }
    return QF_OK;
}

// Group pairs by (class, K).
void add_to_blocks(std::vector<HostBlock>& blocks, int cls, int K, const qf::PairInfo& info, std::vector<double>&& row)
{
    for (auto& b : blocks)
        if (b.cls == cls && b.K == K) {
            b.info.push_back(info);
            b.rows.push_back(std::move(row));
            return;
        }
    HostBlock b;
    b.cls = cls;
    b.K = K;
    b.info.push_back(info);
    b.rows.push_back(std::move(row));
    blocks.push_back(std::move(b));
}

template <class F>
void for_each_canonical_pair(const qf_engine* e, F&& f)
{
    const int nq = (int)e->qs.size();
    for (int a = 0; a < nq; ++a)
        for (int b = 0; b < nq; ++b) {
            const int La = e->qs[a].L, Lb = e->qs[b].L;
            if (La < Lb || (La == Lb && a < b)) continue;
            f(a, b);
        }
}

// Schwarz bounds on the GPU with the diagonal-class kernels:
//   Ycutoff(I,J) = sqrt(max |(ij|ij)|) over the Q-shell pairs of (I,J)
//   cutprim(p,q) = sqrt(X0 * max |(pq|pq)|) for single primitive pairs,
// as QUICK's schwarzoff (quick_cutoff_module.f90:54-588).
int compute_schwarz(qf_engine* e)
{
    e->have_schwarz = false;
    e->ycut.assign((size_t)e->nshell * e->nshell, 0.0);
    e->cutprim.assign((size_t)e->nprim * e->nprim, 0.0);
    for (int pass = 0; pass < 2; ++pass) {
        std::vector<HostBlock> blocks;
        std::vector<int> owner_a, owner_b;   // per block, per pair: Q-shells / prims
        std::vector<std::vector<int>> keys;
        for_each_canonical_pair(e, [&](int a, int b) {
            if (pass == 0) {
                qf::PairInfo info;
                std::vector<double> row;
                int K;
                make_pair(e, a, b, -1, -1, false, info, row, K);
                info.id = a * (int)e->qs.size() + b;
                add_to_blocks(blocks, pair_class(e->qs[a].L, e->qs[b].L), K, info, std::move(row));
            } else {
                for (int i = 0; i < e->qs[a].nprim; ++i)
                    for (int j = 0; j < e->qs[b].nprim; ++j) {
                        qf::PairInfo info;
                        std::vector<double> row;
                        int K;
                        make_pair(e, a, b, i, j, false, info, row, K);
                        info.id = (e->qs[a].pstart + i) * e->nprim + (e->qs[b].pstart + j);
                        add_to_blocks(blocks, pair_class(e->qs[a].L, e->qs[b].L), K, info, std::move(row));
                    }
            }
        });
        DevBuf<qf::PairInfo> dinfo;
        DevBuf<double> dprim;
        std::vector<qf::PairBlock> hb;
        int rc = upload_blocks(e, blocks, dinfo, dprim, hb, 0);
        if (rc) return rc;
        size_t total = 0;
        for (auto& b : blocks) total += b.info.size();
        DevBuf<double> dout;
        QF_HIP(dout.resize(total));
        // global slot buffer of the wave-per-quartet diagonals that need one
        size_t gdoubles = 0;
        for (auto& b : blocks) gdoubles = std::max<size_t>(gdoubles, (size_t)qf::coop_global_doubles(b.cls, b.cls));
        DevBuf<double> dgs;
        if (gdoubles) QF_HIP(dgs.resize(gdoubles * qf::COOP_GLOBAL_SLICES));
        size_t off = 0;
        for (size_t k = 0; k < blocks.size(); ++k) {
            qf::SchwarzLaunch L = qf::schwarz_launcher(blocks[k].cls);
            L(hb[k], dout.p + off, dgs.p, 0);
            off += blocks[k].info.size();
        }
        QF_HIP(hipGetLastError());
        std::vector<double> out(total);
        QF_HIP(hipMemcpy(out.data(), dout.p, total * sizeof(double), hipMemcpyDeviceToHost));
        off = 0;
        for (auto& b : blocks)
            for (auto& info : b.info) {
                const double v = out[off++];
                if (pass == 0) {
                    double& y = e->ycut[(size_t)info.sa * e->nshell + info.sb];
                    y = std::max(y, v);
                    e->ycut[(size_t)info.sb * e->nshell + info.sa] = y;
                } else {
                    const int pa = info.id / e->nprim, pb = info.id % e->nprim;
                    double& c = e->cutprim[(size_t)pa * e->nprim + pb];
                    c = std::max(c, v);
                    e->cutprim[(size_t)pb * e->nprim + pa] = c;
                }
            }
    }
    for (auto& y : e->ycut) y = std::sqrt(y);
    for (auto& c : e->cutprim) c = std::sqrt(kX0 * c);
    e->have_schwarz = true;
    return QF_OK;
}

// For every bra the number of kets with ycut_i*ycut_j > thr (>= where not strict):
// both sorted by ycut descending, so one walk finds them all.
void prefix_counts(const std::vector<qf::PairInfo>& bras, const std::vector<qf::PairInfo>& kets, double thr, bool strict,
                   std::vector<int>& out)
{
    out.resize(bras.size());
    int n = (int)kets.size();
    for (size_t i = 0; i < bras.size(); ++i) {
        while (n > 0) {
            const double y = bras[i].ycut * kets[n - 1].ycut;
            if (strict ? (y > thr) : (y >= thr)) break;
            --n;
        }
        out[i] = n;
    }
}

// Regions of the global slot buffer, one per launch whose node programs keep
// their slots there (launches on different streams run at the same time), of
// one slice per workgroup of its grid.  Returns the doubles needed in all.
size_t slot_doubles(const qf_engine::Launch& L)
{
    return L.tile == 2 ? (size_t)qf::coop_global_doubles(L.cb, L.ck) * std::min(L.count, qf::COOP_GLOBAL_SLICES) : 0;
}

size_t place_slots(std::vector<qf_engine::Launch>& launches)
{
    size_t total = 0;
    for (auto& L : launches) {
        L.gslot = total;
        total += slot_doubles(L);
    }
    return total;
}

// Estimated seconds of a launch: the larger of its longest task alone and all of
// its work spread over the GPU, plus a launch.  Algorithmic FLOPs of every
// quartet of the windows, at 1.3 GFLOP/s for a wave that works through quartets
// one by one ((dd|dd) 39 kFLOP in 34 us, (ff|ff) 340 kFLOP in 476 us) and 0.2
// GFLOP/s for a lane of the per-lane kernels, and at the 1.2 and 6 TFLOP/s that
// whole launches reach.
struct LaunchCost {
    double all = 0.0, longest = 0.0;
    double quartet = 0.0, prim = 0.0;   // FLOPs of the launch that is being added
    bool wave = false;                  // ... and whether it runs a quartet per wave
    void launch(const qf_engine::Launch& L, bool per_wave)
    {
        quartet = qf::class_flops(L.cb, L.ck, 1, 0);
        prim = qf::class_flops(L.cb, L.ck, 0, 1);
        wave = per_wave;
    }
    double task(const qf::Task& k)
    {
        const double one = (quartet + prim * ((k.pe - k.pb) * (k.qe - k.qb))) * (k.ke - k.kb);
        const double t = one * (wave ? k.ket_count / 1.3e9 : 1 / 0.2e9);
        all += one * k.ket_count * (wave ? 1 / 1.2e12 : 1 / 6e12);
        longest = std::max(longest, t);
        return t;
    }
    double seconds() const { return 5e-6 + std::max(longest, all); }
};

// Issue order of launches that take t seconds, and the stream of each: longest
// first, each to the stream with the least time so far.
void stream_order(const std::vector<std::pair<int, double>>& t, qf_engine::Plan& p)
{
    p.order.clear();
    p.gain = 0.0;
    std::vector<int> ord(t.size());
    std::iota(ord.begin(), ord.end(), 0);
    std::stable_sort(ord.begin(), ord.end(), [&](int x, int y) { return t[x].second > t[y].second; });
    double load[kSide + 1] = {};
    for (int l : ord) {
        int to = 0;
        for (int k = 1; k <= kSide; ++k)
            if (load[k] < load[to]) to = k;
        load[to] += t[l].second;
        p.order.push_back({t[l].first, to});
        p.gain += t[l].second;
    }
    p.gain -= *std::max_element(load, load + kSide + 1);
}

void stream_order(const std::vector<qf_engine::Launch>& launches, const std::vector<qf::Task>& tasks,
                  qf_engine::Plan& p)
{
    std::vector<std::pair<int, double>> t;
    for (int l = 0; l < (int)launches.size(); ++l) {
        const auto& L = launches[l];
        LaunchCost c;
        c.launch(L, L.tile == 2);
        for (int x = L.offset; x < L.offset + L.count; ++x) c.task(tasks[x]);
        t.push_back({l, c.seconds()});
    }
    stream_order(t, p);
}

// Molecules whose classes share launches: up to 200 functions, without d shells
// (six classes) up to 100.  Builds in us, one launch per class and stream chain ->
// shared launches (each with the task shapes that suit it): ethane 6-31G (30
// functions) 151 -> 82, glycine 3-21G (55) 143 -> 102, (Gly)2 6-31G (97) 423 -> 434,
// C12H26 6-31G (160) 1027 -> 1107; with d shells water 6-31G* (19) 134 -> 77, ethane
// 6-31G* (42) 273 -> 153, glycine 6-31G** (100) 637 -> 394, ethane def2-TZVP (108, 55
// classes) 1561 -> 1104, (H2O)8 6-31G* (152) 799 -> 526, its cation 1003 -> 679, (Gly)2
// 6-31G** (175) 1411 -> 1373, (H2O)8 cc-pVDZ (200) 1065 -> 960.  Above, a launch
// fills the GPU by itself and a bucket costs its light classes their occupancy:
// (H2O)12 (228) 1484 -> 1513, C20H42 3-21G (264) 911 -> 1097, (H2O)16 (304) 2896 ->
// 2993, (H2O)32 (608) 9982 -> 12755.
bool shares_launches(const qf_engine* e)
{
    int lmax = 0;
    for (int l : e->s_lmax) lmax = std::max(lmax, l);
    return e->tile != 0 && e->nbasis <= (lmax > 1 ? 200 : 100);
}

// Workgroups of a shared launch and their estimated seconds.
struct FusedList {
    std::vector<qf::FusedBlock> blocks;
    std::vector<unsigned short> key;   // exponent and two mantissa bits of the time: steps of at most 25 %
    void add(double t, int cls, int index)
    {
        uint64_t u;
        std::memcpy(&u, &t, sizeof(u));
        blocks.push_back(qf::FusedBlock{cls, index});
        key.push_back((unsigned short)((u >> 50) & 8191));
    }
    // appends them to `out`, longest first (a counting sort: a comparison sort of
    // the 30000 workgroups of a molecule would take longer than its build)
    void append(std::vector<qf::FusedBlock>& out) const
    {
        std::vector<int> at(8193, 0);
        for (unsigned short k : key) ++at[8192 - k];
        for (int k = 1; k <= 8192; ++k) at[k] += at[k - 1];
        const size_t base = out.size();
        out.resize(base + blocks.size());
        for (size_t x = blocks.size(); x-- > 0;) out[base + --at[8192 - key[x]]] = blocks[x];
    }
};

// The kernel that runs a class of closed-shell (os 0) or open-shell (os 1) builds
// beside others (-1: the class has a launch of its own).
int shared_kernel(const qf_engine::Launch& L, int os)
{
    const bool coop = L.tile == 2;
    if (L.fp32 || L.tile == 0 || (os && L.os_split) || (os && !coop && !L.os_lean)) return -1;
    return qf::fuse_bucket(L.cb, L.ck, coop);
}

// Plan of closed-shell (os 0) or open-shell (os 1) builds in which classes of
// the same kernel bucket share a launch, its workgroups longest first.
// Appends to e->fused and to `list`, their workgroups.  Launches run side by side:
// the regions of the shared ones in the global slot buffer follow those of the
// plan's own launches.  Returns the doubles of the buffer that the plan needs.
size_t fuse_plan(qf_engine* e, int os, std::vector<qf::FusedBlock>& list)
{
    struct Group {
        FusedList list;
        LaunchCost cost;
        size_t lds = 0;
    };
    std::map<std::pair<int, int>, Group> groups;   // by kernel and waves
    size_t slots = 0;
    std::vector<std::pair<int, double>> t;
    for (int l = 0; l < (int)e->launches.size(); ++l) {
        const auto& L = e->launches[l];
        const bool coop = L.tile == 2;
        const int id = L.cb * 16 + L.ck;
        const int kernel = shared_kernel(L, os);
        LaunchCost own;
        Group* g = kernel < 0 ? nullptr : &groups[{kernel, coop ? 1 : L.waves}];
        LaunchCost& c = g ? g->cost : own;
        c.launch(L, coop);
        if (g && !coop) {
            const bool two = os && L.lds_os;
            g->lds = std::max(g->lds, two ? L.lds_os : L.lds);
            for (int x = L.goffset; x < L.goffset + L.gcount; ++x) {
                const auto& tg = e->groups[x];
                double wave[4] = {};
                for (int k = tg.task_begin; k < tg.task_end; ++k)
                    wave[(k - tg.task_begin) % L.waves] += c.task(e->tasks[k]);
                g->list.add(*std::max_element(wave, wave + 4), id + (two ? 256 : 0), x);
            }
        } else {
            if (g) g->lds = std::max(g->lds, sizeof(double) * qf::coop_lds_doubles(L.cb, L.ck));
            for (int x = L.offset; x < L.offset + L.count; ++x) {
                const double s = c.task(e->tasks[x]);
                if (g) g->list.add(s, id, x);
            }
        }
        if (!g) {
            t.push_back({l, own.seconds()});
            if (slot_doubles(L)) slots = std::max(slots, L.gslot + slot_doubles(L));
        }
    }
    for (auto& kv : groups) {
        Group& g = kv.second;
        qf_engine::Fused f{};
        f.kernel = kv.first.first;
        f.waves = kv.first.second;
        f.offset = (int)list.size();
        f.count = (int)g.list.blocks.size();
        f.lds = g.lds;
        f.gslot = slots;
        f.seconds = g.cost.seconds();
        slots += (size_t)qf::fuse_kernel(f.kernel).global * std::min(f.count, qf::COOP_GLOBAL_SLICES);
        g.list.append(list);
        t.push_back({~(int)e->fused.size(), f.seconds});
        e->fused.push_back(f);
    }
    stream_order(t, e->plan[os]);
    return slots;
}

// The same for gradients (water 6-31G*, host to host: 291 -> 168 us).
size_t grad_fuse_plan(qf_engine* e, std::vector<qf::FusedBlock>& list)
{
    std::vector<FusedList> lists(qf::kGradFuseKernels);
    std::vector<LaunchCost> cost(qf::kGradFuseKernels);
    std::vector<size_t> lds(qf::kGradFuseKernels, 0);
    std::vector<std::pair<int, double>> t;
    size_t slots = 0;
    for (const auto& L : e->launches) {
        const int k = qf::grad_fuse_bucket(L.cb, L.ck);
        if (k < 0) return 0;   // an f class: gradients are refused
        const bool coop = qf::grad_fuse_kernel(k).coop;
        if (coop) lds[k] = std::max(lds[k], sizeof(double) * qf::grad_lds_doubles(L.cb, L.ck));
        cost[k].launch(L, coop);
        for (int x = L.offset; x < L.offset + L.count; ++x)
            lists[k].add(cost[k].task(e->tasks[x]), L.cb * 16 + L.ck + (L.fp32 ? 256 : 0), x);
    }
    for (int k = 0; k < qf::kGradFuseKernels; ++k) {
        if (lists[k].blocks.empty()) continue;
        qf_engine::Fused f{};
        f.kernel = k;
        f.waves = 1;
        f.offset = (int)list.size();
        f.count = (int)lists[k].blocks.size();
        f.lds = lds[k];
        f.gslot = slots;
        f.seconds = cost[k].seconds();
        slots += (size_t)qf::grad_fuse_kernel(k).global * std::min(f.count, qf::COOP_GLOBAL_SLICES);
        lists[k].append(list);
        t.push_back({~(int)e->fused.size(), f.seconds});
        e->fused.push_back(f);
    }
    stream_order(t, e->plan[2]);
    return slots;
}

// The plan of a build or gradient (kind 2): one launch per class above the sizes of
// shares_launches, where the grid is capped (qf_set_persistent caps each class's) and
// where a gradient kernel was chosen.
const qf_engine::Plan& plan_of(const qf_engine* e, int kind)
{
    bool plain = e->persist > 0 || !e->shared;
    if (kind == 2 && !plain) {
        plain = !e->grad_lane;
        for (const auto& row : e->ctune)
            for (const auto& c : row) plain = plain || c.grad >= 0;
    }
    return e->plan[plain ? 3 : kind];
}

// Primitive pieces: a wave's lanes each run the whole primitive loop of
// one quartet, so the most contracted quartets set the tail of a launch
// (and, for small molecules with few waves, its whole time).  The
// primitive pairs of a task are therefore cut into pieces: a small molecule
// has too few quartets to fill the GPU and takes one primitive pair per
// piece, a large one only cuts the longest loops (e.g. 36 -> 3 x 12), since
// every piece repeats the screen, the HRR and the digestion.  Builds in us
// with pieces of 1 / 2 / 3 / 4 / 6 / 12, launches over four streams:
// water 6-31G* (19 functions) 143 / 184 / 284 / 291 / 396 / 731, butane 6-31G* (80)
// 835 / 521 / 776 / 805 / 1361 / 1793, glycine 6-31G** (100, two tasks a
// workgroup) 1710 / 824 / 614 / 589 / 616 / 989, (H2O)8 6-31G* (152) 1808 /
// 881 / 788 / 857 / 1015 / 1479, (Gly)2 6-31G** (175) 4526 / 2258 / 1483 /
// 1442 / 1560 / 2021, (H2O)16 6-31G* (304) 10064 / 4669 / 2909 / 2823 / 2599 /
// 2931, (H2O)32 (608) 34806 / 17910 / 11420 / 11298 / 10712 / 10692.  Shared
// launches (`shared`) have no tails of their own to shorten and take longer
// pieces; 1 / 2 / 3 / 4 / 6: water 113 / 72 / 91 / - / -, ethane 6-31G* (42) 217 / 151 /
// 255 / 303 / 436, butane 775 / 402 / 357 / 316 / 606, glycine 1116 / 548 / 401 / 393 /
// 436, (H2O)8 6-31G* 1753 / 865 / 587 / 580 / 526, (Gly)2 3839 / 2116 / 1478 / 1472 /
// 1371.  Up to 200 functions the other sizes therefore serve batches (by their
// summed size) and qf_set_tile(0) only, and rest on the single builds above.
// Batches, pieces of 1 / 2 / 3: two molecules 6-31G (size 19) 202 / 104 / 119, 6-31G*
// (26) 287 / 218 / 240, four molecules 3-21G (37) 106 / 130 / 149, three 6-31G* (41)
// 351 / 309 / 417, five 6-31G* (69) 812 / 484 / 529, eight 6-31G (79) 1308 / 543 /
// 394, eight 6-31G* (114) 2180 / 1117 / 896; water 6-31G* without tiles 278 / 210 / -.
// At sizes up to 48 pieces of 2 would serve all of these better but 3-21G.
int prim_piece(const qf_engine* e, int size, bool shared)
{
    return e->prim_piece > 0   ? e->prim_piece
           : e->prim_piece < 0 ? 1 << 20
           : shared            ? (size <= 48 ? 2 : size <= 64 ? 3 : size <= 128 ? 4 : 6)
           : size <= 48        ? 1
           : size <= 96        ? 2
           : size <= 160       ? 3
           : size <= 200       ? 4
           : size <= 400       ? 6
                               : 12;
}

// Kets per task of the wave-per-quartet kernels (builds in us with windows of 1 / 2 / 4 / 8 / 16: (H2O)16 2828 / 2846 /
// 2853 / 2953 / 2987, (H2O)32 10701 / 10658 / 10663 / 11389 / 11136, (Gly)6
// 6-31G** 11829 / 11813 / 12198 / 12191 / 13524)
int coop_window(int size) { return size <= 256 ? 1 : kCoopWindow; }

// A task as tasks of at most `piece` bra and ket primitive pairs each.
template <class F>
void each_piece(qf::Task& t, int Kb, int Kk, int piece, F&& f)
{
    const int nb = (Kb + piece - 1) / piece, nk = (Kk + piece - 1) / piece;
    const int sb = (Kb + nb - 1) / nb, sk = (Kk + nk - 1) / nk;
    for (int pb = 0; pb < Kb; pb += sb)
        for (int qb = 0; qb < Kk; qb += sk) {
            t.pb = pb;
            t.pe = std::min(Kb, pb + sb);
            t.qb = qb;
            t.qe = std::min(Kk, qb + sk);
            f(t);
        }
}

// Work of a task: bras x kets x primitive pairs (bra and ket); without the
// primitive factor the longest-first order misjudges the contracted classes (13 %
// of the (H2O)32 build).
long long task_work(const qf::Task& x)
{
    return (long long)(x.ke - x.kb) * x.ket_count * (x.pe - x.pb) * (x.qe - x.qb);
}

// Indices in order of descending work, equal ones in their order, so that a launch
// ends evenly: by counting, digit by digit.  A comparison sort of the tasks
// themselves was a fifth of prepare.
std::vector<int> longest_first(const std::vector<long long>& work)
{
    const size_t n = work.size();
    std::vector<int> ord(n);
    std::iota(ord.begin(), ord.end(), 0);
    if (n < 512) {
        std::stable_sort(ord.begin(), ord.end(), [&](int x, int y) { return work[x] > work[y]; });
        return ord;
    }
    const long long top = *std::max_element(work.begin(), work.end());
    constexpr int kBits = 11;
    constexpr long long kDigit = (1 << kBits) - 1;
    std::vector<int> next(n);
    for (int shift = 0; shift < 62 && (top >> shift) > 0; shift += kBits) {
        int at[kDigit + 2] = {};
        for (size_t k = 0; k < n; ++k) ++at[kDigit - ((work[k] >> shift) & kDigit) + 1];
        for (int d = 0; d <= kDigit; ++d) at[d + 1] += at[d];
        for (size_t k = 0; k < n; ++k) next[at[kDigit - ((work[ord[k]] >> shift) & kDigit)]++] = ord[k];
        ord.swap(next);
    }
    return ord;
}

template <class T>
void longest_first(T* p, const std::vector<long long>& work)
{
    const std::vector<int> ord = longest_first(work);
    const std::vector<T> was(p, p + ord.size());
    for (size_t k = 0; k < ord.size(); ++k) p[k] = was[ord[k]];
}

void longest_first(std::vector<qf::Task>& tasks, size_t first)
{
    std::vector<long long> work(tasks.size() - first);
    for (size_t x = 0; x < work.size(); ++x) work[x] = task_work(tasks[first + x]);
    longest_first(tasks.data() + first, work);
}

// Tile groups of `groups` from `first` on, by the work of their tasks.
void longest_first(std::vector<qf::TileGroup>& groups, size_t first, const std::vector<qf::Task>& tasks)
{
    std::vector<long long> work(groups.size() - first, 0);
    for (size_t q = 0; q < work.size(); ++q)
        for (int x = groups[first + q].task_begin; x < groups[first + q].task_end; ++x) work[q] += task_work(tasks[x]);
    longest_first(groups.data() + first, work);
}

// How a quartet class runs: the shape of its launch for one precision.
struct ClassShape {
    bool runs = false;       // (the FP32 half of a class that is not split does not)
    int kind;                // 0 direct atomics, 1 LDS tile, 2 one quartet per wave
    bool split, closed_only;
    int mmax, win, piece;    // bras and kets a task, primitive pairs a piece
    int tile_tasks, tile_waves;
};

// `size` stands for the number of basis functions in the rules that choose launch
// shapes: the engine's own, or for an engine in a batch that of the molecule whose
// build holds as much work (the precision split goes by the engine's own size);
// shared: tile and wave-per-quartet classes share launches.
int class_shape(const qf_engine* e, int cb, int ck, int fp32, int size, bool shared, ClassShape& out)
{
    out.runs = false;
    const int na = ncart(kClassL[cb][0]), nb = ncart(kClassL[cb][1]);
    // bras per task: long loops for cheap classes (more register
    // accumulation, fewer atomics), short ones for expensive classes
    // (enough waves to fill 256 CUs)
    const int ni = na * nb * ncart(kClassL[ck][0]) * ncart(kClassL[ck][1]);
    const qf_engine::ClassTune& ct = e->ctune[cb][ck];
    int mmax = ni <= 10 ? 16 : ni <= 36 ? 8 : ni <= 108 ? 4 : ni <= 324 ? 2 : 1;
    // up to 32 functions at most 2 bras per task: more, shorter
    // tasks for launches that hold few (QUICK's regression inputs
    // up to 32 functions, geometric mean 16.3x -> 17.8x QUICK's
    // saved build times; no gain above)
    if (size <= 32) mmax = std::min(mmax, 2);
    if (ct.mmax > 0) mmax = ct.mmax;
    // tasks per tile workgroup: few for small molecules, whose launches
    // hold few tasks (builds in us with 1 / 2 / 4 / 8 / 16: glycine
    // 6-31G** 633 / 633 / 814 / 992 / 992, (H2O)8 6-31G* 924 / 885 / 975 /
    // 928 / 1180, (H2O)8 cc-pVDZ (200 functions) 1077 / 1129 / 1202 / 1242 /
    // 1447, C20H42 3-21G (264) 1825 / 1105 / 912 / 897 / 994, (H2O)16
    // 3703 / 2940 / 3133 / 3171 / 3142, (H2O)32 25512 / 14599 / 12000 / 11245 /
    // 10973; shared launches, 1 / 2 / 4: ethane 6-31G* 155 / 151 / 237, glycine
    // 393 / 442 / 593, (H2O)8 6-31G* 516 / 526 / 628, its cation 853 / 677 / 753,
    // (Gly)2 6-31G** 1438 / 1371 / 1889; between, (H2O)3 6-31G* (57) 275 / 270 / 470,
    // (H2O)4 (76) 327 / 494 / 575, butane (80) 348 / 343 / 581, (H2O)5 (95) 363 / 386 /
    // 577, C5H12 (99) 481 / 497 / 913, (H2O)6 (114) 428 / 425 / 700, C6H14 (118) 617 /
    // 648 / 980; batches, 1 / 2 / 4 / 8: two molecules 6-31G* (size 26) 385 / 296 / 252 /
    // 273, five (69) 477 / 474 / 515 / 591, twelve (186) 1971 / 2202 / 2651 / 2517, 24 (272)
    // 4396 / 4963 / 6236 / 6061: the line at 256 is the single molecules')
    int tile_tasks = ct.tpg > 0        ? ct.tpg
                           : e->tile_tasks > 0 ? e->tile_tasks
                           : shared            ? (size <= 48 || size > 128 ? 2 : 1)
                           : size <= 256       ? 2
                           : size <= 400       ? 4
                                               : 16;
    int tile_waves = ct.waves > 0 ? ct.waves : e->tile_waves;
    // LDS tile: (na + m*nb) x ncol exchange terms + m*na*nb Coulomb terms
    int maxcol = 0;
    for (const auto& Kb : e->blocks)
        if (Kb.cls == ck) maxcol = std::max(maxcol, (int)Kb.colf.size());
    const long long room = e->lds_budget / 8 - (long long)na * maxcol;
    const long long mfit = room > 0 ? room / ((long long)nb * maxcol + na * nb) : 0;
    // Mixed precision splits a class only where its FP32 half can run
    // through the LDS-tile kernel: the direct-atomic FP32 kernels of
    // (dp|dp) gave wrong Fock matrices on gfx950 and the (dd|dp) one
    // non-finite values, while CPU builds of the same code are right.
    // (dd|dp) and (dd|dd) stay FP64 (their FP32 forms spill several KB
    // per lane: little to gain).
    // classes without per-lane kernels (La+Lb+Lc+Ld >= 6) run every
    // quartet in FP64 on the wave-per-quartet kernel
    const bool lane_class = qf::fock_launcher(cb, ck) != nullptr;
    // Classes with La+Lb+Lc+Ld >= split_lmin are split (qf_set_split_classes).
    // FP32 quartets compute their Boys function, exponents and
    // recursions in FP32, which shortens the primitive loop (the
    // FP64 Boys function is most of a light class's work) and halves
    // the registers of the spilling d classes.
    const int Lsum_s = kClassL[cb][0] + kClassL[cb][1] + kClassL[ck][0] + kClassL[ck][1];
    // By default every class above 256 functions, and only the
    // classes with La+Lb+Lc+Ld >= 5 below: a small molecule's
    // light classes hold too few quartets for the second launch
    // to pay (256 batched molecules: 1389 builds/s splitting all,
    // FP64 1432).
    const int lmin = e->split_lmin >= 0 ? e->split_lmin : e->nbasis <= 256 ? 5 : 0;
    const bool f_class = std::max(kClassL[cb][0], kClassL[ck][0]) == 3;   // f classes stay FP64
    const bool split_class = e->prec == QF_PREC_MIXED && mfit >= 1 && lane_class && !f_class &&
                             (ct.split >= 0 ? ct.split == 1 : Lsum_s >= lmin);
    if (fp32 && !split_class) return QF_OK;
    // wave-per-quartet kernel (FP64 launches of classes that have one)
    // wave-per-quartet kernel: where the class tuning asks for it, and by
    // default (unless qf_set_tile turned the shared-memory kernels off)
    // for the d-heavy classes (La+Lb+Lc+Ld >= 6; in launches of one class >= 5 up to 128 functions and >= 4 up to 48,
    // where few waves run and latency decides), whose per-lane
    // kernels spill several KB per lane: one such quartet alone on a
    // lane costs milliseconds, which dominates the build of a small
    // molecule
    const int Lsum = kClassL[cb][0] + kClassL[cb][1] + kClassL[ck][0] + kClassL[ck][1];
    // (QUICK's regression inputs of 49-128 functions run their
    // La+Lb+Lc+Ld = 4 classes faster on the tile kernel: PO4 6-31G*
    // 15.8x -> 18.0x, PSB5 6-31G 26x -> 34x QUICK's build times;
    // up to 48 functions and at 5 the wave-per-quartet kernel wins;
    // in shared launches, with La+Lb+Lc+Ld >= 4 / 5 / 6 on it: water 72 / 79 / 97,
    // ethane 6-31G* 211 / 155 / 151, butane 633 / 336 / 316, glycine 800 / 509 /
    // 393, (H2O)8 6-31G* 972 / 635 / 516; small batches were not measured)
    const int coop_lmin = shared ? (size <= 32 ? 4 : 6) : size <= 48 ? 4 : size <= 128 ? 5 : 6;
    const bool tile_class = qf::fock_tile_launcher(cb, ck) != nullptr;
    const bool tile_ok = tile_class && mfit >= 1;
    // Classes whose FP64 tile kernel runs in Hermite Gaussians: above 256
    // functions it takes over from the wave-per-quartet kernel ((dd|ds),
    // (dd|pp) and (dp|dp) together: (H2O)32 10.65 -> 10.2 ms a build, (Gly)10
    // mixed 29.4 -> 26.0; below, too few quartets fill its waves: glycine
    // 6-31G** 0.63 -> 0.93, (H2O)8 cc-pVDZ 1.08 -> 1.26, which a batch does
    // not change: 48 molecules 16.0 -> 16.9), with two waves,
    // four tasks of one bra a workgroup ((dp|pp), (H2O)32: 10.5 ms against
    // 10.7 with the other classes' shapes).
    // A class without another tile kernel takes this one with tile = 1 on the
    // same condition, else the wave-per-quartet kernel, as saved tables
    // mean it: tile = 1 for these three, wave per quartet -> Hermite, water
    // 0.12 -> 0.24 ms, glycine 0.42 -> 0.96, (H2O)8 6-31G* 0.63 -> 1.36, (H2O)12
    // 1.41 -> 2.32, 256 batched molecules in mixed precision 68.0 -> 71.6, but
    // (H2O)16 (304) 2.83 -> 2.80.
    const bool md = !fp32 && tile_ok && qf::fock_tile_is_md(cb, ck);
    const bool md_shape = md && e->nbasis > 256 && ct.tile < 0 && e->tile != 0;
    if (md_shape && ct.mmax == 0) mmax = 1;
    if (md_shape && ct.tpg == 0 && e->tile_tasks == 0) tile_tasks = 4;
    if (md_shape && ct.waves == 0) tile_waves = std::min(tile_waves, 2);
    const bool want_coop = ct.tile == 2   ? true
                           : ct.tile == 1 ? !lane_class && !(tile_ok && e->nbasis > 256)
                           : ct.tile == 0 || e->tile == 0 ? !lane_class
                           : md_shape ? false
                                      : Lsum >= coop_lmin || (!lane_class && !tile_ok);
    const bool coop = !fp32 && want_coop && qf::fock_coop_launcher(cb, ck) != nullptr;
    if (!coop && !lane_class && !tile_ok) return fail(QF_ERR_STATE, "class has no kernel for its launch");
    const bool tile = !coop && tile_ok && (fp32 || !lane_class || (ct.tile >= 0 ? ct.tile != 0 : e->tile != 0));
    if (tile) mmax = (int)std::min<long long>(mmax, mfit);
    // kets per task: a full wave for the per-lane kernels; for the
    // wave-per-quartet kernel a window (the class tuning's
    // tasks_per_group): small windows give more workgroups to
    // classes with few quartets
    out.win = coop ? (ct.tpg > 0 ? std::min(ct.tpg, qf::WAVE) : coop_window(size)) : qf::WAVE;
    out.piece = ct.piece > 0 ? ct.piece : ct.piece < 0 ? 1 << 20 : prim_piece(e, size, shared);
    out.runs = true;
    out.kind = coop ? 2 : tile ? 1 : 0;
    out.split = split_class;
    out.closed_only = tile && !fp32 && !lane_class;
    out.mmax = mmax;
    out.tile_tasks = tile_tasks;
    out.tile_waves = tile_waves;
    return QF_OK;
}

// Buffers of class_tasks, kept over its calls.
struct TaskScratch {
    std::vector<std::pair<int, int>> chunks;   // bra chunks of a block
    std::vector<int> nall, nhigh, lo, hi;      // kets of each bra of a block, of each of a chunk
};

// Appends the wave tasks and tile groups of one class, precision and engine, whose
// blocks are numbered from `base`; the launch's index ranges are those of the
// vectors (count 0: it has none).  order: longest first (a batch orders over its
// molecules itself).
int class_tasks(const qf_engine* e, int cb, int ck, int fp32, const ClassShape& sh, int base, TaskScratch& sc,
                std::vector<qf::Task>& tasks, std::vector<qf::TileGroup>& groups, qf_stats* stats, bool order,
                qf_engine::Launch& L)
{
    const int offset = (int)tasks.size(), goffset = (int)groups.size();
    const int na = ncart(kClassL[cb][0]), nb = ncart(kClassL[cb][1]);
    const qf_engine::ClassTune& ct = e->ctune[cb][ck];
    size_t lds = 0, lds_os = 0;
    long long group_tasks = 0;
    for (size_t bbk = 0; bbk < e->blocks.size(); ++bbk) {
        const HostBlock& B = e->blocks[bbk];
        if (B.cls != cb) continue;
        for (size_t kbk = 0; kbk < e->blocks.size(); ++kbk) {
            const HostBlock& Kb = e->blocks[kbk];
            if (Kb.cls != ck) continue;
            if (cb == ck && kbk > bbk) continue;
            const bool same = (cb == ck && kbk == bbk);
            prefix_counts(B.info, Kb.info, e->list_cutoff(), true, sc.nall);
            if (sh.split) prefix_counts(B.info, Kb.info, e->split_thr, false, sc.nhigh);
            sc.chunks.clear();
            for (const auto& g : B.groups)
                for (int c0 = g.first; c0 < g.second; c0 += sh.mmax)
                    sc.chunks.push_back({c0, std::min(g.second, c0 + sh.mmax)});
            for (const auto& g : sc.chunks) {
                // per bra of the group: ket range [lo, hi) of this precision
                const int M = g.second - g.first;
                sc.lo.resize(M);
                sc.hi.resize(M);
                int nmax = 0;
                for (int k = 0; k < M; ++k) {
                    const int i = B.bperm[g.first + k];
                    const int n = same ? std::min(sc.nall[i], i + 1) : sc.nall[i];
                    if (!fp32 && stats) stats->n_quartets_bound += n;
                    const int n64 = sh.split ? std::min(n, sc.nhigh[i]) : n;
                    sc.lo[k] = fp32 ? n64 : 0;
                    sc.hi[k] = fp32 ? n : n64;
                    nmax = std::max(nmax, sc.hi[k]);
                }
                const int chunk_first = (int)tasks.size();
                for (int s0 = 0; s0 < nmax; s0 += sh.win) {
                    int kb = -1, ke = -1;
                    for (int k = 0; k < M; ++k)
                        if (sc.lo[k] < sc.hi[k] && sc.lo[k] < s0 + sh.win && sc.hi[k] > s0) {
                            if (kb < 0) kb = k;
                            ke = k + 1;
                        }
                    if (kb < 0) continue;
                    qf::Task t{};
                    t.bra_block = base + (int)bbk;
                    t.kb = g.first + kb;
                    t.ke = g.first + ke;
                    t.ket_block = base + (int)kbk;
                    t.ket_start = s0;
                    t.ket_count = std::min(sh.win, nmax - s0);
                    t.same_block = same ? 1 : 0;
                    t.all_fp64 = sh.split ? 0 : 1;
                    // highly contracted pairs: spread the primitive
                    // pairs of the window over several tasks
                    each_piece(t, B.K, Kb.K, sh.piece, [&](const qf::Task& x) { tasks.push_back(x); });
                }
                if (sh.kind != 1) continue;
                // workgroups of the chunk: consecutive runs of its tasks
                const int chunk_end = (int)tasks.size();
                for (int t0 = chunk_first; t0 < chunk_end; t0 += sh.tile_tasks) {
                    qf::TileGroup tg{};
                    tg.task_begin = t0;
                    tg.task_end = std::min(chunk_end, t0 + sh.tile_tasks);
                    tg.chunk_kb = g.first;
                    tg.nbra = M;
                    groups.push_back(tg);
                    group_tasks += tg.task_end - tg.task_begin;
                }
                if (chunk_end > chunk_first) {
                    const size_t kt = (size_t)(na + M * nb) * Kb.colf.size();
                    lds = std::max(lds, sizeof(double) * (kt + (size_t)M * na * nb));
                    lds_os = std::max(lds_os, sizeof(double) * (2 * kt + (size_t)M * na * nb));
                }
            }
        }
    }
    const int count = (int)tasks.size() - offset;
    const int gcount = (int)groups.size() - goffset;
    if (sh.kind == 1) {
        if (order) longest_first(groups, goffset, tasks);
    } else if (e->shuffle && count > 1) {
        // deterministic permutation first: concurrent waves then hit different kets
        uint64_t st = 0x9E3779B97F4A7C15ull ^ (uint64_t)(cb * 12 + ck * 2 + fp32);
        for (int q = count - 1; q > 0; --q) {
            st ^= st << 13;
            st ^= st >> 7;
            st ^= st << 17;
            const int r = (int)(st % (uint64_t)(q + 1));
            std::swap(tasks[offset + q], tasks[offset + r]);
        }
        if (order) longest_first(tasks, offset);
    }
    L = qf_engine::Launch{};
    L.closed_only = sh.closed_only;
    L.cb = cb;
    L.ck = ck;
    L.fp32 = fp32;
    L.offset = offset;
    L.count = count;
    L.tile = sh.kind;
    L.goffset = goffset;
    L.gcount = gcount;
    L.waves = gcount > 0 ? (int)std::min<long long>(sh.tile_waves,
                                                    std::max<long long>(1, (group_tasks + gcount - 1) / gcount))
                         : 1;
    L.lds = lds;
    L.lds_os = lds_os <= kMaxTileLds ? lds_os : 0;
    L.os_split = ct.os == 1;
    L.os_lean = ct.os == 2 || ct.os < 0;
    if (stats) (fp32 ? stats->n_tasks_fp32 : stats->n_tasks_fp64) += count;
    // every tile workgroup must stay inside its chunk and its LDS allocation
    for (int q = goffset; q < goffset + gcount; ++q) {
        const qf::TileGroup& g = groups[q];
        if (g.task_begin < offset || g.task_end > offset + count || g.task_begin >= g.task_end)
            return fail(QF_ERR_STATE, "tile group outside its launch");
        const qf::Task& t0 = tasks[g.task_begin];
        const size_t need = sizeof(double) * ((size_t)(na + g.nbra * nb) * e->blocks[t0.ket_block - base].colf.size() +
                                              (size_t)g.nbra * na * nb);
        if (need > L.lds) return fail(QF_ERR_STATE, "tile group exceeds its LDS allocation");
        if (L.lds_os && 2 * need - sizeof(double) * (size_t)g.nbra * na * nb > L.lds_os)
            return fail(QF_ERR_STATE, "tile group exceeds its open-shell LDS allocation");
        for (int x = g.task_begin; x < g.task_end; ++x) {
            const qf::Task& t = tasks[x];
            if (t.bra_block != t0.bra_block || t.ket_block != t0.ket_block || t.kb < g.chunk_kb ||
                t.ke > g.chunk_kb + g.nbra || t.kb >= t.ke)
                return fail(QF_ERR_STATE, "tile group mixes chunks");
        }
    }
    return QF_OK;
}

// Tasks, tile groups and launches of the engine, per quartet class and precision.
int make_tasks(qf_engine* e)
{
    e->shared = shares_launches(e);
    e->tasks.clear();
    e->groups.clear();
    e->launches.clear();
    TaskScratch sc;
    for (int cb = 0; cb < kNPC; ++cb)
        for (int ck = 0; ck <= cb; ++ck)
            for (int fp32 = 0; fp32 < 2; ++fp32) {
                ClassShape sh;
                qf_engine::Launch L;
                int rc = class_shape(e, cb, ck, fp32, e->nbasis, e->shared, sh);
                if (rc == QF_OK && sh.runs)
                    rc = class_tasks(e, cb, ck, fp32, sh, 0, sc, e->tasks, e->groups, &e->stats, true, L);
                if (rc) return rc;
                if (sh.runs && L.count > 0) e->launches.push_back(L);
            }
    return QF_OK;
}

// Wave-per-quartet tasks of the closed_only classes, longest first, for open-shell
// builds and gradients.  Every bra alone: its kets make windows of one length and a
// shorter one, so the number of tasks of each amount of work is known beforehand and
// every task goes straight to its place.  Made like the other tasks and sorted, they
// were half of prepare for (Gly)10 6-31G** (0.7 million, 32 MB: 24 -> 50 ms, now 18).
int make_alt_tasks(qf_engine* e)
{
    const int win = coop_window(e->nbasis);
    std::vector<int> nall;
    std::vector<long long> windows(win + 1);   // of a pair of blocks, by length
    // f(blocks, task with the fields that all tasks of the blocks share, kets of each bra in nall)
    auto each_pair = [&](const qf_engine::Launch& L, auto&& f) {
        for (int bb = 0; bb < (int)e->blocks.size(); ++bb)
            for (int kb = 0; kb < (int)e->blocks.size(); ++kb) {
                const HostBlock &B = e->blocks[bb], &K = e->blocks[kb];
                if (B.cls != L.cb || K.cls != L.ck || (L.cb == L.ck && kb > bb)) continue;
                prefix_counts(B.info, K.info, e->list_cutoff(), true, nall);
                if (bb == kb)
                    for (size_t i = 0; i < nall.size(); ++i) nall[i] = std::min(nall[i], (int)i + 1);
                qf::Task t{};
                t.bra_block = bb;
                t.ke = 1;
                t.ket_block = kb;
                t.same_block = bb == kb;
                t.all_fp64 = 1;
                f(B, K, t);
            }
    };
    auto piece_of = [&](const qf_engine::Launch& L) {
        const int ct = e->ctune[L.cb][L.ck].piece;
        return ct > 0 ? ct : ct < 0 ? 1 << 20 : prim_piece(e, e->nbasis, e->shared);
    };
    // tasks of each amount of work, the largest first, then the place of the next one
    std::vector<std::map<long long, int, std::greater<long long>>> place(e->launches.size());
    int total = 0;
    for (size_t l = 0; l < e->launches.size(); ++l) {
        auto& L = e->launches[l];
        if (!L.closed_only) continue;
        each_pair(L, [&](const HostBlock& B, const HostBlock& K, qf::Task t) {
            std::fill(windows.begin(), windows.end(), 0);
            for (int n : nall) {
                windows[win] += n / win;
                ++windows[n % win];
            }
            for (t.ket_count = 1; t.ket_count <= win; ++t.ket_count)
                if (const int n = (int)windows[t.ket_count])
                    each_piece(t, B.K, K.K, piece_of(L), [&](const qf::Task& x) { place[l][task_work(x)] += n; });
        });
        L.alt_offset = total;
        for (auto& w : place[l]) {
            const int n = w.second;
            w.second = total;
            total += n;
        }
        L.alt_count = total - L.alt_offset;
    }
    std::unique_ptr<qf::Task[]> tasks(new qf::Task[total]);
    std::vector<std::vector<std::pair<qf::Task, int*>>> pieces(win + 1);   // of a window, by its length
    for (size_t l = 0; l < e->launches.size(); ++l)
        if (e->launches[l].closed_only)
            each_pair(e->launches[l], [&](const HostBlock& B, const HostBlock& K, qf::Task t) {
                for (t.ket_count = 1; t.ket_count <= win; ++t.ket_count) {
                    pieces[t.ket_count].clear();
                    each_piece(t, B.K, K.K, piece_of(e->launches[l]),
                               [&](const qf::Task& x) { pieces[t.ket_count].push_back({x, &place[l][task_work(x)]}); });
                }
                for (int x = 0; x < (int)B.bperm.size(); ++x)
                    for (int k0 = 0, n = nall[B.bperm[x]]; k0 < n; k0 += win)
                        for (auto& p : pieces[std::min(win, n - k0)]) {
                            qf::Task& to = tasks[(*p.second)++];
                            to = p.first;
                            to.kb = x;
                            to.ke = x + 1;
                            to.ket_start = k0;
                        }
            });
    QF_HIP(e->d_alt.resize(total));
    if (total) QF_HIP(hipMemcpy(e->d_alt.p, tasks.get(), total * sizeof(qf::Task), hipMemcpyHostToDevice));
    return QF_OK;
}

// Tasks of a class for its wave-per-quartet kernels.
struct WaveTasks {
    const qf::Task* p;
    int count;
};
WaveTasks wave_tasks(const qf_engine* e, const qf_engine::Launch& L)
{
    if (L.closed_only) return {e->d_alt.p + L.alt_offset, L.alt_count};
    return {e->d_tasks.p + L.offset, L.count};
}

int prepare(qf_engine* e)
{
    if (e->prepared) return QF_OK;   // idempotent: setters clear the flag
    if (e->nshell == 0 || e->natom == 0) return fail(QF_ERR_STATE, "molecule and basis must be set");
    int rc = e->set_device();
    if (rc) return rc;
    if (!e->have_schwarz) {
        rc = compute_schwarz(e);
        if (rc) return rc;
    }
    double ymax = 0.0;
    for (double y : e->ycut) ymax = std::max(ymax, y);

    // ---- pair blocks: canonical pairs that can meet some partner -----------
    e->blocks.clear();
    int next_id = 0;
    for_each_canonical_pair(e, [&](int a, int b) {
        const double y = e->ycut[(size_t)e->qs[a].shell * e->nshell + e->qs[b].shell];
        if (!(y * ymax > e->list_cutoff())) return;
        qf::PairInfo info;
        std::vector<double> row;
        int K;
        make_pair(e, a, b, -1, -1, true, info, row, K);
        info.id = next_id++;
        add_to_blocks(e->blocks, pair_class(e->qs[a].L, e->qs[b].L), K, info, std::move(row));
    });
    // order: by class, then K; pairs inside a block by ycut descending
    std::sort(e->blocks.begin(), e->blocks.end(),
              [](const HostBlock& x, const HostBlock& y) { return x.cls != y.cls ? x.cls < y.cls : x.K < y.K; });
    for (auto& b : e->blocks) {
        std::vector<size_t> ord(b.info.size());
        std::iota(ord.begin(), ord.end(), 0);
        std::stable_sort(ord.begin(), ord.end(), [&](size_t x, size_t y) { return b.info[x].ycut > b.info[y].ycut; });
        std::vector<qf::PairInfo> info2;
        std::vector<std::vector<double>> rows2;
        for (size_t k : ord) {
            info2.push_back(b.info[k]);
            rows2.push_back(std::move(b.rows[k]));
        }
        b.info.swap(info2);
        b.rows.swap(rows2);
    }
    for (auto& b : e->blocks) {
        // bra order: grouped by first Q-shell a, Schwarz-descending inside a group
        const int nb = (int)b.info.size();
        b.bperm.resize(nb);
        std::iota(b.bperm.begin(), b.bperm.end(), 0);
        std::stable_sort(b.bperm.begin(), b.bperm.end(),
                         [&](int x, int y) { return b.info[x].qa < b.info[y].qa; });
        b.groups.clear();
        for (int k = 0; k < nb;) {
            int e2 = k;
            while (e2 < nb && b.info[b.bperm[e2]].qa == b.info[b.bperm[k]].qa) ++e2;
            b.groups.push_back({k, e2});
            k = e2;
        }
    }
    for (auto& b : e->blocks) {
        // compact columns: the functions of every Q-shell of the block, by Q-shell id
        std::vector<int> qlist;
        for (const auto& p : b.info) {
            qlist.push_back(p.qa);
            qlist.push_back(p.qb);
        }
        std::sort(qlist.begin(), qlist.end());
        qlist.erase(std::unique(qlist.begin(), qlist.end()), qlist.end());
        std::vector<int> qcol(e->qs.size(), -1);
        b.colf.clear();
        for (int q : qlist) {
            qcol[q] = (int)b.colf.size();
            for (int f = 0; f < ncart(e->qs[q].L); ++f) b.colf.push_back(e->qs[q].fn + f);
        }
        for (auto& p : b.info) {
            p.cola = qcol[p.qa];
            p.colb = qcol[p.qb];
        }
    }
    rc = upload_blocks(e, e->blocks, e->d_info, e->d_prim, e->hblocks, 0, &e->d_perm, &e->d_colf);
    if (rc) return rc;
    for (auto& b : e->blocks) b.rows.clear();
    QF_HIP(e->d_blocks.upload(e->hblocks));

    // ---- wave tasks per quartet class and precision ------------------------
    e->split_thr = e->split * ymax * ymax;
    e->stats = qf_stats{};
    for (auto& b : e->blocks) e->stats.n_pairs += (long long)b.info.size();
    rc = make_tasks(e);
    if (rc) return rc;
    QF_HIP(e->d_tasks.upload(e->tasks));
    QF_HIP(e->d_groups.upload(e->groups));
    if ((rc = make_alt_tasks(e))) return rc;
    e->drop_replays();
    // global slot buffer of the wave-per-quartet classes that keep their
    // node-program slots in global memory
    size_t gdoubles = place_slots(e->launches);
    e->fused.clear();
    e->grad_slots = 0;
    stream_order(e->launches, e->tasks, e->plan[3]);
    if (e->shared) {
        std::vector<qf::FusedBlock> list;
        for (int os = 0; os < 2; ++os) gdoubles = std::max(gdoubles, fuse_plan(e, os, list));
        e->grad_slots = grad_fuse_plan(e, list);
        QF_HIP(e->d_fused.upload(list));
    }
    if (gdoubles) QF_HIP(e->d_cscratch.resize(gdoubles));

    // ---- per-build buffers -------------------------------------------------
    const size_t n2 = (size_t)e->nbasis * e->nbasis;
    QF_HIP(e->d_Gt.resize(n2 * e->replicas));
    QF_HIP(e->d_Gs.resize(n2));
    QF_HIP(e->d_P.resize(n2));
    QF_HIP(e->d_cm.resize((size_t)e->nshell * e->nshell));
    std::vector<int> shells(3 * (size_t)e->nshell);
    for (int k = 0; k < e->nshell; ++k) {
        int nf = 0;
        for (int L = e->s_lmin[k]; L <= e->s_lmax[k]; ++L) nf += ncart(L);
        shells[k] = e->s_fstart[k];
        shells[e->nshell + k] = e->s_fstart[k] + nf - 1;
        shells[2 * e->nshell + k] = e->s_atom[k];
    }
    QF_HIP(e->d_shells.upload(shells));
    QF_HIP(e->d_mol.resize(4));   // slots: build / open-shell pass 1, open-shell pass 2, no-alloc build, gradient
    QF_HIP(e->d_counts.resize(2 * std::max<size_t>(1, e->launches.size())));
    e->stats.device_bytes = (long long)(e->d_info.bytes() + e->d_prim.bytes() + e->d_tasks.bytes() + e->d_alt.bytes() +
                                        e->d_Gt.bytes() * 3 + e->d_cm.bytes() + e->d_blocks.bytes());
    // launch indices recorded for timing refer to the old launch list
    e->ev_used = 0;
    e->ev_launch.clear();
    e->built = false;
    e->count_cm_own = false;
    e->grad_built = false;
    e->grad_cm_own = false;
    ++e->generation;
    e->prepared = true;
    return QF_OK;
}

// Fixed scratch of qf_fock_build_device_noalloc: G partials, symmetrised G
// and the Cutmatrix of one build live here instead of in buffers the
// library allocates.  Each device holds its own copy for the life of the
// process.  Host code never passes `scratch` itself to a kernel (on the host
// it names a stand-in, not device memory): it uses the address
// hipGetSymbolAddress returns, looked up once per device in
// qf_engine_create with that device current.
constexpr size_t kNoAllocDoubles = QF_NOALLOC_SCRATCH_BYTES / sizeof(double);
__device__ __align__(256) double scratch[kNoAllocDoubles];

constexpr int kMaxDevices = 64;
double* g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mu;

int noalloc_scratch_init(int device)
{
    if (device < 0 || device >= kMaxDevices) return fail(QF_ERR_BADDEVICE, "device id beyond the no-alloc table");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return QF_OK;
    int prev = 0;
    if (hipGetDevice(&prev) != hipSuccess) return fail(QF_ERR_NODEVICE, "hipGetDevice");
    if (hipSetDevice(device) != hipSuccess) return fail(QF_ERR_BADDEVICE, "hipSetDevice");
    void* p = nullptr;
    const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    (void)hipSetDevice(prev);
    if (err != hipSuccess || !p) return fail(QF_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(err));
    g_scratch_ptr[device] = static_cast<double*>(p);
    return QF_OK;
}

double* noalloc_scratch_ptr(int device)
{
    if (device < 0 || device >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return g_scratch_ptr[device];
}

// One pass over every class launch: G(P) with the density screen dcm, then
// F += G.  `slot` picks the
// device MolDesc, so two passes can be queued back to back on one stream.
// Where a build keeps G: `replicas` copies of nbasis^2 at Gt (the atomics'
// targets) and the symmetrised G at Gs.  The engine's own buffers, or the
// fixed scratch array of the no-alloc entry point.
struct GBufs {
    double* Gt;
    int replicas;
    double* Gs;
    bool timing;   // per-launch HIP events (never in the no-alloc path: it creates events)
    bool fork;     // side streams and replay (not in the no-alloc path: they allocate)
    double* Gt2 = nullptr;   // open-shell pass: accumulators of the second exchange density
    // densities in host memory, copied to Pc and Pd, and host memory for the result
    const double *hP = nullptr, *hQ = nullptr;
    double *Pc = nullptr, *Pd = nullptr, *H = nullptr, *H2 = nullptr;
};

// Issues the launches of `order` with issue(launch index, stream): forked
// from s over the side streams and joined again, or all on s where there are
// none.  After a failed launch or event call every side stream that took part is
// joined all the same, so that a capture of s stays whole and what follows on s
// waits for the launches that were made; the first error is returned.
template <class F>
int issue_forked(SideStreams* side, hipStream_t s, const std::vector<std::pair<int, int>>& order, F&& issue)
{
    int rc = QF_OK;
    if (!side || !side_free(*side, s)) {
        for (const auto& o : order)
            if ((rc = issue(o.first, s))) return rc;
        return rc;
    }
    auto ok = [&](hipError_t err, const char* call) {
        if (err == hipSuccess) return true;
        if (rc == QF_OK) rc = fail(QF_ERR_HIP, std::string(call) + ": " + hipGetErrorString(err));
        return false;
    };
    bool used[kSide] = {};
    QF_HIP(hipEventRecord(side->fork, s));
    for (const auto& o : order) {
        hipStream_t q = s;
        if (o.second > 0) {
            q = side->s[o.second - 1];
            if (!used[o.second - 1]) {
                if (!ok(hipStreamWaitEvent(q, side->fork, 0), "hipStreamWaitEvent(fork)")) break;
                used[o.second - 1] = true;
            }
        }
        if ((rc = issue(o.first, q))) break;
    }
    for (int k = 0; k < kSide; ++k)
        if (used[k] && ok(hipEventRecord(side->done[k], side->s[k]), "hipEventRecord(done)"))
            ok(hipStreamWaitEvent(s, side->done[k], 0), "hipStreamWaitEvent(done)");
    return rc;
}

// Records the start event of a timed launch; *stop is the event that ends it.
int timing_begin(qf_engine* e, int li, hipStream_t s, hipEvent_t* stop)
{
    while (e->ev_pool.size() < e->ev_used + 2) {
        hipEvent_t ev;
        QF_HIP(hipEventCreate(&ev));
        e->ev_pool.push_back(ev);
    }
    QF_HIP(hipEventRecord(e->ev_pool[e->ev_used], s));
    *stop = e->ev_pool[e->ev_used + 1];
    e->ev_used += 2;
    e->ev_launch.push_back(li);
    return QF_OK;
}

// Issues one kind of build (0 closed shell, 1 open shell, 2 gradient): the
// opening kernel, the class launches by issue(launch index, target) and the
// closing kernel (none where close is null).  The first build since a prepare
// is issued launch by launch, the classes forked over the side streams where
// that saves more than its ten event calls cost (about 60 us).  From the second
// on it is replayed from a graph of the same four chains; of its arguments
// only those of the opening and closing kernels change (densities and results
// reach the class kernels through the descriptor that the opening kernel
// writes).  What bounds a small build is host time and the waits between
// streams.  Device builds, us, one stream / forked launches / replay: water
// STO-3G 73 / 94 / 72, water 6-31G* 314 / 217 / 132, glycine 6-31G** 1497 / 1018 /
// 670, ethane def2-TZVP 4482 / 2498 / 1568.  A build under capture is issued
// launch by launch.
template <class F>
int issue_build(qf_engine* e, int kind, hipStream_t s, const OpenArgs& open, const CloseArgs* close, F&& issue)
{
    Replay& r = e->replay[kind];
    const bool captured = is_capturing(s);
    const qf_engine::Plan& plan = plan_of(e, kind);
    if (!captured && r.old.size() >= 4) r.sweep();
    if (!captured && !r.exec && !r.failed && !plan.order.empty() && ++r.uses > 1) {
        hipGraphNode_t last[kSide + 1] = {};
        bool ok = hipGraphCreate(&r.graph, 0) == hipSuccess;
        if (ok) {
            qf::LaunchTo to(r.graph, nullptr, 0);
            open_build(open, to);
            r.first = to.node;
            ok = to.err == hipSuccess;
        }
        for (const auto& o : plan.order) {
            if (!ok) break;
            qf::LaunchTo to(r.graph, last[o.second] ? &last[o.second] : &r.first, 1);
            const int rc = issue(o.first, to);
            if (rc) {
                r.drop();
                return rc;
            }
            last[o.second] = to.node;
            ok = to.err == hipSuccess;
        }
        if (ok && close) {
            hipGraphNode_t ends[kSide + 1];
            int n = 0;
            for (auto x : last)
                if (x) ends[n++] = x;
            qf::LaunchTo to(r.graph, ends, n);
            close_build(*close, to);
            r.last = to.node;
            ok = to.err == hipSuccess;
        }
        ok = ok && hipGraphInstantiate(&r.exec, r.graph, nullptr, nullptr, 0) == hipSuccess;
        if (ok) {
            r.open = open;
            if (close) r.close = *close;
        } else {
            (void)hipGetLastError();
            r.drop();
            r.failed = true;
        }
    }
    if (!captured && r.exec) {
        if (std::memcmp(&r.open, &open, sizeof(open))) {
            qf::LaunchTo to(r.exec, r.first);
            open_build(open, to);
            QF_HIP(to.err);
            r.open = open;
        }
        if (close && std::memcmp(&r.close, close, sizeof(*close))) {
            qf::LaunchTo to(r.exec, r.last);
            close_build(*close, to);
            QF_HIP(to.err);
            r.close = *close;
        }
        QF_HIP(hipGraphLaunch(r.exec, s));
        return QF_OK;
    }
    qf::LaunchTo to(s);
    open_build(open, to);
    const bool forked = plan.order.size() > 1 && (e->side || plan.gain > 8e-5) && side_ready(e->side, e->device, s);
    const int rc = issue_forked(forked ? e->side : nullptr, s, plan.order, [&](int li, hipStream_t q) {
        qf::LaunchTo x(q);
        return issue(li, x);
    });
    if (rc) return rc;
    if (close) close_build(*close, to);
    return QF_OK;
}

// cm_out: where the opening kernel puts the density screen matrix (null: dcm
// is the caller's).  dPb != nullptr: the open-shell pass.  Every integral is
// digested with dP (Coulomb and exchange, into Gt) and with the spin density
// dP2 (exchange only, into gb.Gt2);
// then dF += A + B and dF2 += A - B (k_close).  A class with os_split
// runs as two closed-shell launches instead of the fused one: dP into Gt,
// then dP2 with a zero Coulomb density (e->d_zero) into Gt2 (descriptor slot
// 1).
int build_pass(qf_engine* e, const double* dP, const double* dcm, double* dF, int slot, hipStream_t s,
               const GBufs& gb, double* cm_out, const double* dPa = nullptr, const double* dPb = nullptr,
               double* dF2 = nullptr)
{
    // open shell: dPa and dPb are the caller's densities, dP the engine's total
    // density and e->d_Ps its spin density, both computed by the opening kernel
    const int os = dPb != nullptr;
    const double* dP2 = os ? e->d_Ps.p : nullptr;
    if (os && (!gb.Gt2 || (!gb.H && (!dF || !dF2)) || !e->d_zero.p)) return fail(QF_ERR_ARG, "open-shell pass without its buffers");
    const int n = e->nbasis, ns = e->nshell;
    qf::MolDesc md{};
    md.P = dP;
    md.PJ = dP;
    md.G = gb.Gt;
    md.cutmat = dcm;
    md.nbasis = n;
    md.nshell = ns;
    md.cutoff = e->cutoff;
    md.primlim = e->primlim;
    md.hyb = e->hyb;
    md.replicas = gb.replicas;
    md.split = (e->prec == QF_PREC_MIXED) ? e->split_thr : 0.0;
    md.P2 = dP2;
    md.G2 = gb.Gt2;
    qf::MolDesc* dmol = e->d_mol.p + slot;
    qf::MolDesc* dmol_x = nullptr;   // exchange-only pass of the two-pass open-shell classes
    OpenArgs oa{};
    oa.md = md;
    oa.dmd = dmol;
    if (os) {
        oa.mx = md;
        oa.mx.P = dP2;
        oa.mx.PJ = e->d_zero.p;
        oa.mx.G = gb.Gt2;
        oa.mx.P2 = nullptr;
        oa.mx.G2 = nullptr;
        oa.dmx = dmol_x = e->d_mol.p + 1;
        oa.Pt = e->d_Pt.p;
        oa.Ps = e->d_Ps.p;
    }
    oa.Pa = gb.hP ? gb.hP : os ? dPa : dP;
    oa.Pb = gb.hP ? gb.hQ : dPb;
    oa.Pc = gb.Pc;
    oa.Pd = gb.Pd;
    oa.G = gb.Gt;
    oa.G2 = os ? gb.Gt2 : nullptr;
    oa.ng = (size_t)n * n * gb.replicas;
    oa.cm = cm_out;
    oa.f0 = e->shell_f0();
    oa.f1 = e->shell_f1();
    oa.n = n;
    oa.nshell = ns;
    CloseArgs ca{};
    ca.Gt = gb.Gt;
    ca.Gt2 = os ? gb.Gt2 : nullptr;
    ca.Gs = gb.Gs;
    ca.F = dF;
    ca.F2 = os ? dF2 : nullptr;
    ca.H = gb.H;
    ca.H2 = gb.H2;
    ca.replicas = gb.replicas;
    ca.n = n;
    // one class launch with descriptor m on stream q; los: its open-shell form
    auto launch = [&](const qf_engine::Launch& L, qf::MolDesc* m, int los, qf::LaunchTo& q) -> int {
        if (L.tile == 2 || (los && L.closed_only)) {
            qf::FockCoopLaunch fc = qf::fock_coop_launcher(L.cb, L.ck);
            if (!fc) return fail(QF_ERR_ARG, "no wave-per-quartet kernel for class");
            const WaveTasks w = wave_tasks(e, L);
            fc(w.p, w.count, e->d_blocks.p, m, los, e->persist, e->d_cscratch.p + L.gslot, q);
        } else if (L.tile) {
            qf::FockTileLaunch ft = qf::fock_tile_launcher(L.cb, L.ck);
            if (!ft) return fail(QF_ERR_ARG, "no tile kernel for class");
            // open shell: a second exchange tile where two fit, else its terms go to Gt2
            const int tos = !los ? 0 : L.lds_os ? 1 : 2;
            ft(e->d_groups.p + L.goffset, L.gcount, e->d_tasks.p, e->d_blocks.p, m, L.fp32,
               tos | (los && L.os_lean ? 4 : 0), L.waves, tos == 1 ? L.lds_os : L.lds, e->persist, q);
        } else {
            qf::FockLaunch f = qf::fock_launcher(L.cb, L.ck);
            if (!f) return fail(QF_ERR_ARG, "no per-lane kernel for class");
            if (f(e->d_tasks.p + L.offset, L.count, e->d_blocks.p, m, L.fp32, los, e->persist, q))
                return fail(QF_ERR_ARG, kDirectFp32Refused);
        }
        return QF_OK;
    };
    auto class_launch = [&](const qf_engine::Launch& L, qf::LaunchTo& q) -> int {
        if (!(os && L.os_split)) return launch(L, dmol, os, q);
        const int rc = launch(L, dmol, 0, q);
        return rc ? rc : launch(L, dmol_x, 0, q);
    };
    auto shared_launch = [&](const qf_engine::Fused& f, qf::LaunchTo& q) -> int {
        qf::fuse_kernel(f.kernel).launch(e->d_fused.p + f.offset, f.count, e->d_groups.p, e->d_tasks.p, e->d_blocks.p,
                                         dmol, os, f.waves, f.lds, e->d_cscratch.p + f.gslot, q);
        return QF_OK;
    };
    if (gb.fork && !gb.timing) {
        const int rc = issue_build(e, os, s, oa, &ca,
                                   [&](int li, qf::LaunchTo& q) {
                                       return li < 0 ? shared_launch(e->fused[~li], q)
                                                     : class_launch(e->launches[li], q);
                                   });
        if (rc) return rc;
    } else if (!gb.timing) {
        // one after another on s
        qf::LaunchTo to(s);
        open_build(oa, to);
        for (const auto& o : plan_of(e, os).order) {
            const int rc = o.first < 0 ? shared_launch(e->fused[~o.first], to) : class_launch(e->launches[o.first], to);
            if (rc) return rc;
        }
        close_build(ca, to);
    } else {
        // class by class between events
        qf::LaunchTo to(s);
        open_build(oa, to);
        for (size_t li = 0; li < e->launches.size(); ++li) {
            hipEvent_t eb = nullptr;
            if (timing_begin(e, (int)li, s, &eb)) return QF_ERR_HIP;
            const int rc = class_launch(e->launches[li], to);
            if (rc) return rc;
            QF_HIP(hipEventRecord(eb, s));
        }
        close_build(ca, to);
    }
    QF_HIP(hipGetLastError());
    return QF_OK;
}

int build(qf_engine* e, const double* dP, double* dF, const double* dcm, hipStream_t s, double* stage = nullptr)
{
    if (!e->prepared) return fail(QF_ERR_STATE, "qf_prepare has not been called");
    double* cm_out = dcm ? nullptr : e->d_cm.p;
    if (!dcm) dcm = cm_out;
    GBufs gb{e->d_Gt.p, e->replicas, e->d_Gs.p, e->timing, true};
    if (stage) {
        gb.hP = stage;
        gb.Pc = e->d_P.p;
        gb.H = stage + (size_t)e->nbasis * e->nbasis;
    }
    const int rc = build_pass(e, dP, dcm, dF, 0, s, gb, cm_out);
    if (rc == QF_OK) {
        e->built = true;
        e->count_cm_own = (dcm == e->d_cm.p);
    }
    return rc;
}

// Open-shell build (QUICK's get_oshell_eri, gpu_get2e_subs.h OSHELL
// branches): Fa += J(Pt) - hyb K(Pa), Fb += J(Pt) - hyb K(Pb).  With the
// spin density Ps = Pa - Pb:
//   A = J(Pt) - hyb/2 K(Pt)   (the closed-shell G of Pt)
//   B = -hyb/2 K(Ps)          (exchange terms only)
// and Fa += A + B, Fb += A - B.  One pass computes each integral once and
// digests it with both densities (the OS kernel instantiations); it screens
// with QUICK's open-shell density matrix, so it sees exactly the quartets
// QUICK's kernel sees.
int build_os(qf_engine* e, const double* dPa, const double* dPb, double* dFa, double* dFb, const double* dcm,
             hipStream_t s, double* stage = nullptr)
{
    if (!e->prepared) return fail(QF_ERR_STATE, "qf_prepare has not been called");
    const int n2 = e->nbasis * e->nbasis;
    QF_HIP(e->d_Pt.resize(n2));
    QF_HIP(e->d_Ps.resize(n2));
    double* cm_out = dcm ? nullptr : e->d_cm.p;
    if (!dcm) dcm = cm_out;
    QF_HIP(e->d_Gt2.resize((size_t)n2 * e->replicas));
    if (e->d_zero.n < (size_t)n2) {
        QF_HIP(e->d_zero.resize(n2));
        hipLaunchKernelGGL(k_zero, dim3(256), dim3(256), 0, s, e->d_zero.p, (size_t)n2);
    }
    GBufs gb{e->d_Gt.p, e->replicas, e->d_Gs.p, e->timing, true};
    gb.Gt2 = e->d_Gt2.p;
    if (stage) {
        gb.hP = stage;
        gb.hQ = stage + n2;
        gb.Pc = e->d_P.p;
        gb.Pd = e->d_Pb.p;
        gb.H = stage + 2 * n2;
        gb.H2 = stage + 3 * n2;
    }
    const int rc = build_pass(e, e->d_Pt.p, dcm, dFa, 0, s, gb, cm_out, dPa, dPb, dFb);
    if (rc == QF_OK) {
        e->built = true;
        e->count_cm_own = (dcm == e->d_cm.p);
    }
    return rc;
}

}  // namespace

// ==========================================================================
// C ABI
// ==========================================================================
extern "C" {

const char* qf_last_error(void) { return g_err.c_str(); }

int qf_engine_create(int device, qf_engine** out)
{
    if (!out) return fail(QF_ERR_ARG, "out is NULL");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count == 0) return fail(QF_ERR_NODEVICE, "no GPU visible");
    if (device < 0) {
        if (hipGetDevice(&device) != hipSuccess) return fail(QF_ERR_NODEVICE, "hipGetDevice");
    }
    if (device >= count) return fail(QF_ERR_BADDEVICE, "device id out of range");
    const int rc = noalloc_scratch_init(device);
    if (rc) return rc;
    qf_engine* e = new qf_engine();
    e->device = device;
    *out = e;
    return QF_OK;
}

void qf_engine_destroy(qf_engine* e)
{
    if (!e) return;
    (void)hipSetDevice(e->device);
    delete e;
}

int qf_set_molecule(qf_engine* e, int natom, const double* xyz)
{
    if (!e || natom <= 0 || !xyz) return fail(QF_ERR_ARG, "bad molecule");
    e->natom = natom;
    e->xyz.assign(xyz, xyz + 3 * natom);
    e->prepared = false;
    e->have_schwarz = false;
    return QF_OK;
}

int qf_set_basis(qf_engine* e, int nshell, const int* shell_atom, const int* shell_lmin, const int* shell_lmax,
                 const int* shell_nprim, const int* shell_pstart, const int* shell_fstart, int nprim_total,
                 const double* exps, const double* coef, int nbasis)
{
    if (!e || nshell <= 0 || nprim_total <= 0 || nbasis <= 0) return fail(QF_ERR_ARG, "bad basis sizes");
    for (int s = 0; s < nshell; ++s) {
        if (shell_lmin[s] < 0 || shell_lmax[s] > 3 || shell_lmin[s] > shell_lmax[s])
            return fail(QF_ERR_ARG, "angular momentum above f is not supported");
        if (shell_atom[s] < 0 || shell_atom[s] >= e->natom) return fail(QF_ERR_ARG, "shell atom out of range");
        if (shell_pstart[s] < 0 || shell_pstart[s] + shell_nprim[s] > nprim_total || shell_nprim[s] <= 0)
            return fail(QF_ERR_ARG, "shell primitive range out of range");
        int nf = 0;
        for (int L = shell_lmin[s]; L <= shell_lmax[s]; ++L) nf += ncart(L);
        if (shell_fstart[s] < 0 || shell_fstart[s] + nf > nbasis) return fail(QF_ERR_ARG, "function range");
    }
    e->nshell = nshell;
    e->nprim = nprim_total;
    e->nbasis = nbasis;
    e->s_atom.assign(shell_atom, shell_atom + nshell);
    e->s_lmin.assign(shell_lmin, shell_lmin + nshell);
    e->s_lmax.assign(shell_lmax, shell_lmax + nshell);
    e->s_nprim.assign(shell_nprim, shell_nprim + nshell);
    e->s_pstart.assign(shell_pstart, shell_pstart + nshell);
    e->s_fstart.assign(shell_fstart, shell_fstart + nshell);
    e->exps.assign(exps, exps + nprim_total);
    e->coef.assign(coef, coef + 4 * (size_t)nprim_total);
    build_qshells(e);
    e->prepared = false;
    e->have_schwarz = false;
    return QF_OK;
}

int qf_set_cutoffs(qf_engine* e, double integral_cutoff, double prim_limit, double hyb)
{
    if (!e || !(integral_cutoff > 0) || !(prim_limit > 0)) return fail(QF_ERR_ARG, "cutoffs must be > 0");
    e->cutoff = integral_cutoff;
    e->primlim = prim_limit;
    e->hyb = hyb;
    e->prepared = false;
    return QF_OK;
}

int qf_set_precision(qf_engine* e, int mode, double split)
{
    if (!e || (mode != QF_PREC_FP64 && mode != QF_PREC_MIXED) || !(split > 0)) return fail(QF_ERR_ARG, "precision");
    e->prec = mode;
    e->split = split;
    e->prepared = false;
    return QF_OK;
}

int qf_set_split_classes(qf_engine* e, int min_lsum)
{
    if (!e || min_lsum < -1) return fail(QF_ERR_ARG, "min_lsum must be >= -1");
    e->split_lmin = min_lsum;
    e->prepared = false;
    return QF_OK;
}

int qf_set_class_split(qf_engine* e, int cb, int ck, int mode)
{
    if (!e) return fail(QF_ERR_ARG, "NULL");
    if (cb < 0 || cb >= kNPC || ck < 0 || ck > cb) return fail(QF_ERR_ARG, "class index out of range");
    if (mode < -1 || mode > 1) return fail(QF_ERR_ARG, "mode must be -1, 0 (FP64) or 1 (split)");
    e->ctune[cb][ck].split = mode;
    e->prepared = false;
    return QF_OK;
}

int qf_set_schwarz(qf_engine* e, const double* ycutoff, const double* cutprim)
{
    if (!e || e->nshell == 0) return fail(QF_ERR_STATE, "set the basis first");
    e->prepared = false;
    if (!ycutoff || !cutprim) {
        e->have_schwarz = false;
        int rc = e->set_device();
        return rc ? rc : compute_schwarz(e);
    }
    e->ycut.assign(ycutoff, ycutoff + (size_t)e->nshell * e->nshell);
    e->cutprim.assign(cutprim, cutprim + (size_t)e->nprim * e->nprim);
    e->have_schwarz = true;
    return QF_OK;
}

int qf_get_schwarz(qf_engine* e, double* ycutoff, double* cutprim)
{
    if (!e || !e->have_schwarz) return fail(QF_ERR_STATE, "no Schwarz bounds yet");
    if (ycutoff) std::memcpy(ycutoff, e->ycut.data(), e->ycut.size() * sizeof(double));
    if (cutprim) std::memcpy(cutprim, e->cutprim.data(), e->cutprim.size() * sizeof(double));
    return QF_OK;
}

int qf_prepare(qf_engine* e)
{
    if (!e) return fail(QF_ERR_ARG, "engine is NULL");
    return prepare(e);
}

int qf_get_stats(qf_engine* e, qf_stats* out)
{
    if (!e || !out) return fail(QF_ERR_ARG, "NULL");
    *out = e->stats;
    return QF_OK;
}

int qf_fock_build_device(qf_engine* e, const double* d_P, double* d_F, const double* d_cutmat, void* stream)
{
    if (!e || !d_P) return fail(QF_ERR_ARG, "NULL");
    int rc = e->set_device();
    if (rc) return rc;
    return build(e, d_P, d_F, d_cutmat, (hipStream_t)stream);
}

int qf_fock_build_device_noalloc(qf_engine* e, const double* d_P, double* d_F, const double* d_cutmat, void* stream)
{
    if (!e || !d_P) return fail(QF_ERR_ARG, "NULL");
    int rc = e->set_device();
    if (rc) return rc;
    if (!e->prepared) return fail(QF_ERR_STATE, "qf_prepare has not been called");
    double* base = noalloc_scratch_ptr(e->device);
    if (!base) return fail(QF_ERR_STATE, "no-alloc scratch not set up on this device");
    const size_t n2 = (size_t)e->nbasis * e->nbasis, ns2 = (size_t)e->nshell * e->nshell;
    if (2 * n2 + (d_cutmat ? 0 : ns2) > (size_t)kNoAllocDoubles)
        return fail(QF_ERR_ARG, "no-alloc build: nbasis too large for the fixed scratch (2 nbasis^2 + nshell^2 "
                                "doubles must fit in QF_NOALLOC_SCRATCH_BYTES)");
    for (const auto& L : e->launches)
        if (L.tile == 2 && qf::coop_global_doubles(L.cb, L.ck) > 0)
            return fail(QF_ERR_ARG, "no-alloc build: a class keeps its node-program slots in global memory");
    const hipStream_t s = (hipStream_t)stream;
    // scratch layout: [G partials n^2 | symmetrised G n^2 | Cutmatrix nshell^2]
    double* Gt = base;
    double* Gs = base + n2;
    double* cm_out = d_cutmat ? nullptr : base + 2 * n2;
    if (!d_cutmat) d_cutmat = cm_out;
    return build_pass(e, d_P, d_cutmat, d_F, 2, s, GBufs{Gt, 1, Gs, false, false}, cm_out);
}

// Two-electron gradient (QUICK's gpu_get_cshell_eri_grad_ -> getGrad,
// gpu_get2e.cu:695-725): one wave-per-quartet gradient launch per class
// over the tasks of the Fock build's launches (their union covers every
// quartet in both precision halves), screened with gradCutoff.
namespace {
constexpr size_t kGradLdsMax = 64 * 1024;   // dynamic LDS of one gradient workgroup

int grad_pass(qf_engine* e, const double* dP, const double* dcm, double* cm_out, double* dgrad, hipStream_t s,
              const double* hP = nullptr)
{
    // every class needs a gradient kernel: check before launching anything
    auto lane_kernel = [&](const qf_engine::Launch& L) -> qf::GradLaunch {
        const int gm = e->ctune[L.cb][L.ck].grad;
        return (gm >= 0 ? gm == 1 : e->grad_lane) ? qf::grad_lane_launcher(L.cb, L.ck) : nullptr;
    };
    for (const auto& L : e->launches)
        if (!qf::grad_launcher(L.cb, L.ck))
            return fail(QF_ERR_ARG, "ERI gradients cover shells up to d; this basis has f shells");
    size_t gdoubles = 0;
    std::vector<size_t> gslot;   // per launch: its region of the global slot buffer
    for (const auto& L : e->launches) {
        gslot.push_back(gdoubles);
        if (!lane_kernel(L))
            gdoubles += (size_t)qf::grad_global_doubles(L.cb, L.ck) *
                        std::min(wave_tasks(e, L).count, qf::COOP_GLOBAL_SLICES);
    }
    gdoubles = std::max(gdoubles, e->grad_slots);
    if (gdoubles && e->d_gscratch.n < gdoubles) {
        e->replay[2].drop();   // it holds the old buffer
        QF_HIP(e->d_gscratch.resize(gdoubles));
    }
    qf::MolDesc md{};
    md.P = dP;
    md.PJ = dP;
    md.G = nullptr;
    md.cutmat = dcm;
    md.nbasis = e->nbasis;
    md.nshell = e->nshell;
    md.cutoff = e->grad_cutoff > 0.0 ? e->grad_cutoff : e->cutoff;
    md.primlim = e->primlim;
    md.hyb = e->hyb;
    md.split = (e->prec == QF_PREC_MIXED) ? e->split_thr : 0.0;   // only separates the launches' halves
    md.replicas = 1;
    md.natom = e->natom;
    md.shell_atom = e->shell_at();
    md.grad = dgrad;
    qf::MolDesc* dmol = e->d_mol.p + 3;
    OpenArgs oa{};
    oa.md = md;
    oa.dmd = dmol;
    oa.Pa = dP;
    if (hP) {                // density in host memory, gradient buffer to be cleared
        oa.Pa = hP;
        oa.Pc = e->d_P.p;
        oa.G = dgrad;
        oa.ng = (size_t)3 * e->natom;
    }
    oa.cm = cm_out;
    oa.f0 = e->shell_f0();
    oa.f1 = e->shell_f1();
    oa.n = e->nbasis;
    oa.nshell = e->nshell;
    const size_t tile_bytes = (size_t)3 * e->natom * sizeof(double);
    auto launch = [&](int li, qf::LaunchTo& q) -> int {
        if (li < 0) {
            const qf_engine::Fused& f = e->fused[~li];
            qf::grad_fuse_kernel(f.kernel).launch(e->d_fused.p + f.offset, f.count, e->d_tasks.p, e->d_blocks.p, dmol,
                                                  (int)(f.lds / sizeof(double)),
                                                  f.lds + tile_bytes <= kGradLdsMax ? 3 * e->natom : 0,
                                                  e->d_gscratch.p + f.gslot, q);
            return QF_OK;
        }
        const auto& L = e->launches[li];
        const qf::GradLaunch lane = lane_kernel(L);
        const size_t slots = lane ? 0 : (size_t)qf::grad_lds_doubles(L.cb, L.ck) * sizeof(double);
        const size_t tile = slots + tile_bytes <= kGradLdsMax ? tile_bytes : 0;
        // one workgroup per task unless the engine caps the grid (qf_set_persistent):
        // the hardware then hands out tasks as workgroups finish
        const WaveTasks w = wave_tasks(e, L);
        const int grid = e->persist > 0 ? std::min(w.count, e->persist) : w.count;
        (lane ? lane : qf::grad_launcher(L.cb, L.ck))(w.p, w.count, e->d_blocks.p, dmol, grid, tile,
                                                      e->d_gscratch.p + gslot[li], L.fp32, q);
        return QF_OK;
    };
    if (!e->timing) {
        const int rc = issue_build(e, 2, s, oa, nullptr, launch);
        if (rc) return rc;
    } else {
        qf::LaunchTo to(s);
        open_build(oa, to);
        for (size_t li = 0; li < e->launches.size(); ++li) {
            hipEvent_t eb = nullptr;
            if (timing_begin(e, (int)li, s, &eb)) return QF_ERR_HIP;
            launch((int)li, to);
            QF_HIP(hipEventRecord(eb, s));
        }
    }
    QF_HIP(hipGetLastError());
    return QF_OK;
}
}  // namespace

int qf_set_grad_cutoff(qf_engine* e, double grad_cutoff)
{
    if (!e || !(grad_cutoff > 0.0)) return fail(QF_ERR_ARG, "gradient cutoff must be positive");
    const double before = e->list_cutoff();
    e->grad_cutoff = grad_cutoff;
    if (e->list_cutoff() != before) e->prepared = false;   // the lists must reach further down
    return QF_OK;
}

int qf_set_grad_kernel(qf_engine* e, int lane)
{
    if (!e) return fail(QF_ERR_ARG, "engine is NULL");
    e->grad_lane = lane != 0;
    e->replay[2].retire();
    return QF_OK;
}

int qf_set_grad_class(qf_engine* e, int cb, int ck, int mode)
{
    if (!e) return fail(QF_ERR_ARG, "engine is NULL");
    if (cb < 0 || cb >= kNPC || ck < 0 || ck > cb) return fail(QF_ERR_ARG, "class index out of range");
    if (mode < -1 || mode > 1) return fail(QF_ERR_ARG, "mode must be -1, 0 (wave-per-quartet) or 1 (per-lane)");
    e->ctune[cb][ck].grad = mode;
    e->replay[2].retire();
    return QF_OK;
}

static int eri_grad(qf_engine* e, const double* d_P, double* d_grad, const double* d_cutmat, hipStream_t s,
                    const double* hP = nullptr)
{
    double* cm_out = d_cutmat ? nullptr : e->d_cm.p;
    const double* dcm = d_cutmat ? d_cutmat : cm_out;
    const int rc = grad_pass(e, d_P, dcm, cm_out, d_grad, s, hP);
    if (rc == QF_OK) {
        e->grad_built = true;
        e->grad_cm_own = (dcm == e->d_cm.p);
    }
    return rc;
}

int qf_eri_grad_device(qf_engine* e, const double* d_P, double* d_grad, const double* d_cutmat, void* stream)
{
    if (!e || !d_P || !d_grad) return fail(QF_ERR_ARG, "NULL");
    int rc = e->set_device();
    if (rc) return rc;
    if (!e->prepared) return fail(QF_ERR_STATE, "qf_prepare has not been called");
    return eri_grad(e, d_P, d_grad, d_cutmat, (hipStream_t)stream);
}

int qf_eri_grad_host(qf_engine* e, const double* P, double* grad, const double* cutmat)
{
    if (!e || !P || !grad) return fail(QF_ERR_ARG, "NULL");
    int rc = e->set_device();
    if (rc) return rc;
    if (!e->prepared) return fail(QF_ERR_STATE, "qf_prepare has not been called");
    const size_t n2 = (size_t)e->nbasis * e->nbasis, ng = (size_t)3 * e->natom;
    if (e->d_grad.n < ng) QF_HIP(e->d_grad.resize(ng));
    Stage stage(n2 + ng);
    if (stage.p) {
        std::memcpy(stage.p, P, n2 * sizeof(double));
    } else {
        QF_HIP(hipMemcpy(e->d_P.p, P, n2 * sizeof(double), hipMemcpyHostToDevice));
        QF_HIP(hipMemset(e->d_grad.p, 0, ng * sizeof(double)));
    }
    const double* dcm = nullptr;
    if (cutmat) {
        QF_HIP(hipMemcpy(e->d_cm.p, cutmat, (size_t)e->nshell * e->nshell * sizeof(double), hipMemcpyHostToDevice));
        dcm = e->d_cm.p;
    }
    rc = eri_grad(e, e->d_P.p, e->d_grad.p, dcm, nullptr, stage.p);
    if (rc) return rc;
    std::vector<double> g(stage.p ? 0 : ng);
    if (stage.p) {
        hipLaunchKernelGGL(k_copy, dim3((ng + 255) / 256), dim3(256), 0, 0, e->d_grad.p, stage.p + n2, (int)ng);
        QF_HIP(hipGetLastError());
        if ((rc = stage.wait())) return rc;
    } else {
        QF_HIP(hipMemcpy(g.data(), e->d_grad.p, ng * sizeof(double), hipMemcpyDeviceToHost));
    }
    const double* got = stage.p ? stage.p + n2 : g.data();
    for (size_t k = 0; k < ng; ++k) grad[k] += got[k];
    return QF_OK;
}

int qf_grad_launch_flops(qf_engine* e, double* flops, long long* quartets, long long* prims)
{
    // counts, with the density screen of the last gradient, the quartets and
    // primitive quartets the gradient launches evaluate, priced with the
    // generated per-class gradient FLOP table
    if (!e || !e->prepared) return fail(QF_ERR_STATE, "not prepared");
    if (!e->grad_built) return fail(QF_ERR_STATE, "no gradient since the last qf_prepare");
    if (!e->grad_cm_own)
        return fail(QF_ERR_STATE, "the last gradient screened with a caller-owned Cutmatrix; counts need one that "
                                  "computes its own (d_cutmat = NULL)");
    int rc = e->set_device();
    if (rc) return rc;
    const size_t nl = e->launches.size();
    QF_HIP(hipMemset(e->d_counts.p, 0, 2 * std::max<size_t>(nl, 1) * sizeof(unsigned long long)));
    for (size_t k = 0; k < nl; ++k) {
        const auto& L = e->launches[k];
        hipLaunchKernelGGL(k_count, dim3(L.count), dim3(qf::WAVE), 0, 0, e->d_tasks.p + L.offset, L.count,
                           e->d_blocks.p, e->d_mol.p + 3, e->d_counts.p, (int)k, L.fp32, 1);
    }
    QF_HIP(hipGetLastError());
    std::vector<unsigned long long> c(2 * std::max<size_t>(nl, 1));
    QF_HIP(hipMemcpy(c.data(), e->d_counts.p, c.size() * sizeof(unsigned long long), hipMemcpyDeviceToHost));
    for (size_t k = 0; k < nl; ++k) {
        if (flops) flops[k] = qf::grad_class_flops(e->launches[k].cb, e->launches[k].ck, c[2 * k], c[2 * k + 1]);
        if (quartets) quartets[k] = (long long)c[2 * k];
        if (prims) prims[k] = (long long)c[2 * k + 1];
    }
    return QF_OK;
}

int qf_fock_build_host(qf_engine* e, const double* P, double* F, const double* cutmat)
{
    if (!e || !P || !F) return fail(QF_ERR_ARG, "NULL");
    int rc = e->set_device();
    if (rc) return rc;
    if (!e->prepared) return fail(QF_ERR_STATE, "qf_prepare has not been called");
    const size_t n2 = (size_t)e->nbasis * e->nbasis;
    Stage stage(2 * n2);
    if (stage.p)
        std::memcpy(stage.p, P, n2 * sizeof(double));
    else
        QF_HIP(hipMemcpy(e->d_P.p, P, n2 * sizeof(double), hipMemcpyHostToDevice));
    const double* dcm = nullptr;
    if (cutmat) {
        QF_HIP(hipMemcpy(e->d_cm.p, cutmat, (size_t)e->nshell * e->nshell * sizeof(double), hipMemcpyHostToDevice));
        dcm = e->d_cm.p;
    }
    rc = build(e, e->d_P.p, nullptr, dcm, 0, stage.p);
    if (rc) return rc;
    if (stage.p) {
        if ((rc = stage.wait())) return rc;
        for (size_t k = 0; k < n2; ++k) F[k] += stage.p[n2 + k];
        return QF_OK;
    }
    std::vector<double> G(n2);
    QF_HIP(hipMemcpy(G.data(), e->d_Gs.p, n2 * sizeof(double), hipMemcpyDeviceToHost));
    for (size_t k = 0; k < n2; ++k) F[k] += G[k];
    return QF_OK;
}

int qf_fock_build_os_device(qf_engine* e, const double* d_Pa, const double* d_Pb, double* d_Fa, double* d_Fb,
                            const double* d_cutmat, void* stream)
{
    if (!e || !d_Pa || !d_Pb || !d_Fa || !d_Fb) return fail(QF_ERR_ARG, "NULL");
    int rc = e->set_device();
    if (rc) return rc;
    return build_os(e, d_Pa, d_Pb, d_Fa, d_Fb, d_cutmat, (hipStream_t)stream);
}

int qf_fock_build_os_host(qf_engine* e, const double* Pa, const double* Pb, double* Fa, double* Fb,
                          const double* cutmat)
{
    if (!e || !Pa || !Pb || !Fa || !Fb) return fail(QF_ERR_ARG, "NULL");
    int rc = e->set_device();
    if (rc) return rc;
    if (!e->prepared) return fail(QF_ERR_STATE, "qf_prepare has not been called");
    const size_t n2 = (size_t)e->nbasis * e->nbasis;
    QF_HIP(e->d_Pb.resize(n2));
    QF_HIP(e->d_Fa.resize(n2));
    QF_HIP(e->d_Fb.resize(n2));
    Stage stage(4 * n2);
    if (stage.p) {
        std::memcpy(stage.p, Pa, n2 * sizeof(double));
        std::memcpy(stage.p + n2, Pb, n2 * sizeof(double));
    } else {
        QF_HIP(hipMemcpy(e->d_P.p, Pa, n2 * sizeof(double), hipMemcpyHostToDevice));
        QF_HIP(hipMemcpy(e->d_Pb.p, Pb, n2 * sizeof(double), hipMemcpyHostToDevice));
        QF_HIP(hipMemcpy(e->d_Fa.p, Fa, n2 * sizeof(double), hipMemcpyHostToDevice));
        QF_HIP(hipMemcpy(e->d_Fb.p, Fb, n2 * sizeof(double), hipMemcpyHostToDevice));
    }
    const double* dcm = nullptr;
    if (cutmat) {
        QF_HIP(hipMemcpy(e->d_cm.p, cutmat, (size_t)e->nshell * e->nshell * sizeof(double), hipMemcpyHostToDevice));
        dcm = e->d_cm.p;
    }
    rc = stage.p ? build_os(e, e->d_P.p, e->d_Pb.p, nullptr, nullptr, dcm, 0, stage.p)
                 : build_os(e, e->d_P.p, e->d_Pb.p, e->d_Fa.p, e->d_Fb.p, dcm, 0);
    if (rc) return rc;
    if (stage.p) {
        if ((rc = stage.wait())) return rc;
        for (size_t k = 0; k < n2; ++k) {
            Fa[k] += stage.p[2 * n2 + k];
            Fb[k] += stage.p[3 * n2 + k];
        }
        return QF_OK;
    }
    QF_HIP(hipMemcpy(Fa, e->d_Fa.p, n2 * sizeof(double), hipMemcpyDeviceToHost));
    QF_HIP(hipMemcpy(Fb, e->d_Fb.p, n2 * sizeof(double), hipMemcpyDeviceToHost));
    return QF_OK;
}

const double* qf_device_g(qf_engine* e) { return e ? e->d_Gs.p : nullptr; }

int qf_internal_basis(qf_engine* e, int* natom, const double** xyz, int* nshell, const int** s_atom,
                      const int** s_lmin, const int** s_lmax, const int** s_nprim, const int** s_pstart,
                      const int** s_fstart, int* nprim, const double** exps, const double** coef, int* nbasis)
{
    if (!e || e->nshell == 0 || e->natom == 0) return fail(QF_ERR_STATE, "molecule and basis must be set");
    int rc = e->set_device();
    if (rc) return rc;
    *natom = e->natom;
    *xyz = e->xyz.data();
    *nshell = e->nshell;
    *s_atom = e->s_atom.data();
    *s_lmin = e->s_lmin.data();
    *s_lmax = e->s_lmax.data();
    *s_nprim = e->s_nprim.data();
    *s_pstart = e->s_pstart.data();
    *s_fstart = e->s_fstart.data();
    *nprim = e->nprim;
    *exps = e->exps.data();
    *coef = e->coef.data();
    *nbasis = e->nbasis;
    return QF_OK;
}

double qf_flops_estimate(qf_engine* e)
{
    const int n = qf_launch_count(e);
    if (n < 0) return -1.0;
    std::vector<double> f(std::max(n, 1));
    if (qf_launch_flops(e, f.data()) != QF_OK) return -1.0;
    double tot = 0.0;
    for (int k = 0; k < n; ++k) tot += f[k];
    e->flops_last = tot;
    return tot;
}

int qf_launch_count(qf_engine* e)
{
    if (!e || !e->prepared) return -1;
    return (int)e->launches.size();
}

int qf_launch_info(qf_engine* e, int idx, int* cb, int* ck, int* fp32, int* ntasks)
{
    if (!e || !e->prepared || idx < 0 || idx >= (int)e->launches.size()) return fail(QF_ERR_ARG, "launch index");
    const auto& L = e->launches[idx];
    *cb = L.cb;
    *ck = L.ck;
    *fp32 = L.fp32;
    *ntasks = L.count;
    return QF_OK;
}

int qf_launch_flops(qf_engine* e, double* flops)
{
    // Counts, with the density of the last build, the quartets and primitive
    // quartets that pass the screens in every launch, and prices them with
    // the generated per-class FLOP table.
    // The kernel reads the screen settings and the Cutmatrix of the last
    // build (device MolDesc slot 0), so it needs a build since the last
    // prepare, screened with the engine's own Cutmatrix (a caller-owned one
    // may be gone by now).
    if (!e || !e->prepared) return fail(QF_ERR_STATE, "not prepared");
    if (!e->built) return fail(QF_ERR_STATE, "no Fock build since the last qf_prepare: counts use its density screen");
    if (!e->count_cm_own)
        return fail(QF_ERR_STATE, "the last build screened with a caller-owned Cutmatrix; counts need a build "
                                  "that computes its own (d_cutmat = NULL)");
    int rc = e->set_device();
    if (rc) return rc;
    const size_t nl = e->launches.size();
    QF_HIP(hipMemset(e->d_counts.p, 0, 2 * std::max<size_t>(nl, 1) * sizeof(unsigned long long)));
    for (size_t k = 0; k < nl; ++k) {
        const auto& L = e->launches[k];
        hipLaunchKernelGGL(k_count, dim3(L.count), dim3(qf::WAVE), 0, 0, e->d_tasks.p + L.offset, L.count,
                           e->d_blocks.p, e->d_mol.p, e->d_counts.p, (int)k, L.fp32, 0);
    }
    QF_HIP(hipGetLastError());
    std::vector<unsigned long long> c(2 * std::max<size_t>(nl, 1));
    QF_HIP(hipMemcpy(c.data(), e->d_counts.p, c.size() * sizeof(unsigned long long), hipMemcpyDeviceToHost));
    for (size_t k = 0; k < nl; ++k) flops[k] = qf::class_flops(e->launches[k].cb, e->launches[k].ck, c[2 * k], c[2 * k + 1]);
    return QF_OK;
}

int qf_launch_counts(qf_engine* e, long long* quartets, long long* prims)
{
    if (!e || !e->prepared) return fail(QF_ERR_STATE, "not prepared");
    const size_t nl = e->launches.size();
    std::vector<double> tmp(std::max<size_t>(nl, 1));
    int rc = qf_launch_flops(e, tmp.data());
    if (rc) return rc;
    std::vector<unsigned long long> c(2 * std::max<size_t>(nl, 1));
    QF_HIP(hipMemcpy(c.data(), e->d_counts.p, c.size() * sizeof(unsigned long long), hipMemcpyDeviceToHost));
    for (size_t k = 0; k < nl; ++k) {
        quartets[k] = (long long)c[2 * k];
        prims[k] = (long long)c[2 * k + 1];
    }
    return QF_OK;
}

int qf_set_tuning(qf_engine* e, int replicas, int shuffle)
{
    if (!e || replicas < 1 || replicas > 256) return fail(QF_ERR_ARG, "replicas must be in 1..256");
    e->replicas = replicas;
    e->shuffle = shuffle != 0;
    e->prepared = false;
    return QF_OK;
}

int qf_set_tile(qf_engine* e, int enable, int waves, int tasks_per_group, int lds_bytes)
{
    if (!e) return fail(QF_ERR_ARG, "NULL");
    if (waves < 1 || waves > 4) return fail(QF_ERR_ARG, "waves must be in 1..4");
    if (tasks_per_group < 0) return fail(QF_ERR_ARG, "tasks_per_group must be >= 0 (0: automatic)");
    if (lds_bytes < 1024 || lds_bytes > 64 * 1024) return fail(QF_ERR_ARG, "lds_bytes must be in 1 KiB..64 KiB");
    e->tile = enable != 0;
    e->tile_waves = waves;
    e->tile_tasks = tasks_per_group;
    e->lds_budget = lds_bytes;
    e->prepared = false;
    return QF_OK;
}

int qf_set_class_tuning(qf_engine* e, int cb, int ck, int tile, int waves, int tasks_per_group, int bras_per_task)
{
    if (!e) return fail(QF_ERR_ARG, "NULL");
    if (cb < 0 || cb >= kNPC || ck < 0 || ck > cb) return fail(QF_ERR_ARG, "class index out of range");
    if (waves > 4 || bras_per_task > 64) return fail(QF_ERR_ARG, "waves <= 4 and bras_per_task <= 64");
    qf_engine::ClassTune& t = e->ctune[cb][ck];
    if (tile > 2) return fail(QF_ERR_ARG, "tile must be -1, 0 (direct), 1 (LDS tile) or 2 (wave per quartet)");
    t.tile = tile < 0 ? -1 : tile;
    t.waves = std::max(0, waves);
    t.tpg = std::max(0, tasks_per_group);
    t.mmax = std::max(0, bras_per_task);
    e->prepared = false;
    return QF_OK;
}

int qf_set_class_os(qf_engine* e, int cb, int ck, int mode)
{
    if (!e) return fail(QF_ERR_ARG, "NULL");
    if (cb < 0 || cb >= kNPC || ck < 0 || ck > cb) return fail(QF_ERR_ARG, "class index out of range");
    if (mode < -1 || mode > 2) return fail(QF_ERR_ARG, "mode must be -1, 0 (fused), 1 (two passes) or 2 (fused lean)");
    e->ctune[cb][ck].os = mode;
    e->prepared = false;
    return QF_OK;
}

int qf_set_class_piece(qf_engine* e, int cb, int ck, int piece)
{
    if (!e) return fail(QF_ERR_ARG, "NULL");
    if (cb < 0 || cb >= kNPC || ck < 0 || ck > cb) return fail(QF_ERR_ARG, "class index out of range");
    e->ctune[cb][ck].piece = piece;
    e->prepared = false;
    return QF_OK;
}

int qf_set_prim_split(qf_engine* e, int piece)
{
    if (!e) return fail(QF_ERR_ARG, "NULL");
    e->prim_piece = piece;
    e->prepared = false;
    return QF_OK;
}

int qf_set_persistent(qf_engine* e, int max_workgroups)
{
    if (!e || max_workgroups < 0) return fail(QF_ERR_ARG, "max_workgroups must be >= 0");
    e->persist = max_workgroups;
    for (auto& r : e->replay) r.retire();
    return QF_OK;
}

int qf_set_timing(qf_engine* e, int enable)
{
    if (!e) return fail(QF_ERR_ARG, "NULL");
    e->timing = enable != 0;
    e->ev_used = 0;
    e->ev_launch.clear();
    return QF_OK;
}

int qf_read_timing(qf_engine* e, double* ms_per_launch, int* calls_per_launch)
{
    // Sums the event-measured duration of every recorded class launch since
    // the last read, per launch index; waits for the last recorded event.
    if (!e || !e->prepared) return fail(QF_ERR_STATE, "not prepared");
    const size_t nl = e->launches.size();
    for (size_t k = 0; k < nl; ++k) {
        ms_per_launch[k] = 0.0;
        calls_per_launch[k] = 0;
    }
    if (e->ev_used) QF_HIP(hipEventSynchronize(e->ev_pool[e->ev_used - 1]));
    for (size_t r = 0; r < e->ev_launch.size(); ++r) {
        if (e->ev_launch[r] < 0 || (size_t)e->ev_launch[r] >= nl) continue;
        float ms = 0.0f;
        QF_HIP(hipEventElapsedTime(&ms, e->ev_pool[2 * r], e->ev_pool[2 * r + 1]));
        ms_per_launch[e->ev_launch[r]] += ms;
        calls_per_launch[e->ev_launch[r]] += 1;
    }
    e->ev_used = 0;
    e->ev_launch.clear();
    return QF_OK;
}

}  // extern "C"

// ==========================================================================
// Batches: many prepared engines (molecules) built together, one launch per
// quartet class for all of them, optionally replayed from a HIP graph.
// Each molecule keeps its own pair data (owned by its engine); the batch
// owns the combined block/task/group tables and pooled P, F, G and Cutmatrix
// buffers, so every pointer a launch uses is fixed and the whole build can be
// captured once and replayed.
// ==========================================================================
namespace {

struct BatchMol {
    const double* P;
    double* F;
    double* Gt;      // replicas * n * n
    double* Gs;      // n * n
    double* cm;      // ns * ns
    const int* f0;
    const int* f1;
    int n, ns;
};

__global__ void k_cutmat_batch(const BatchMol* __restrict__ bm)
{
    const BatchMol m = bm[blockIdx.y];
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= m.ns * m.ns) return;
    const int I = idx / m.ns, J = idx % m.ns;
    double v = 0.0;
    for (int i = m.f0[I]; i <= m.f1[I]; ++i)
        for (int j = m.f0[J]; j <= m.f1[J]; ++j) v = fmax(v, fabs(m.P[i * m.n + j]));
    m.cm[idx] = v;
}

__global__ void k_clear_batch(const BatchMol* __restrict__ bm)
{
    const BatchMol m = bm[blockIdx.y];
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < m.n * m.n) m.F[idx] = 0.0;
}

__global__ void k_add(double* __restrict__ y, const double* __restrict__ x, int count)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < count) y[idx] += x[idx];
}

__global__ void k_finalize_batch(const BatchMol* __restrict__ bm, int replicas)
{
    const BatchMol m = bm[blockIdx.y];
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= m.n * m.n) return;
    const int i = idx / m.n, j = idx % m.n;
    const size_t n2 = (size_t)m.n * m.n;
    double g = 0.0;
    for (int r = 0; r < replicas; ++r) g += m.Gt[r * n2 + i * m.n + j] + m.Gt[r * n2 + j * m.n + i];
    m.Gs[idx] = g;
    m.F[idx] += g;
}

}  // namespace

struct qf_batch {
    int device = 0;
    std::vector<qf_engine*> engs;
    std::vector<unsigned long long> gens;   // each engine's generation when the batch copied its tables
    int replicas = 2;
    int persist = 0;
    std::vector<qf_engine::Launch> launches;
    std::vector<BatchMol> mols;
    DevBuf<BatchMol> d_bm;
    DevBuf<qf::PairBlock> d_blocks;
    DevBuf<qf::Task> d_tasks;
    DevBuf<qf::TileGroup> d_groups;
    DevBuf<qf::MolDesc> d_moldesc;
    DevBuf<double> d_P, d_F, d_Gt, d_Gs, d_cm;
    DevBuf<double> d_cscratch;   // global slots of the wave-per-quartet classes that need them
    size_t gt_total = 0;
    int max_n2 = 0, max_ns2 = 0;
    // graph replay
    bool use_graph = false;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hipStream_t cap_stream = nullptr;
    // per-launch timing (eager builds only)
    bool timing = false;
    std::vector<hipEvent_t> ev_pool;
    size_t ev_used = 0;
    std::vector<int> ev_launch;
    std::vector<std::pair<int, int>> order;   // issue order: (launch index, stream 0..kSide)
    SideStreams* side = nullptr;
    ~qf_batch()
    {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        if (cap_stream) (void)hipStreamDestroy(cap_stream);
        SidePool::get().give(side);
        for (hipEvent_t ev : ev_pool) (void)hipEventDestroy(ev);
    }
};

namespace {

int batch_issue(qf_batch* b, hipStream_t s)
{
    const int nm = (int)b->mols.size();
    hipLaunchKernelGGL(k_cutmat_batch, dim3((b->max_ns2 + 255) / 256, nm), dim3(256), 0, s, b->d_bm.p);
    hipLaunchKernelGGL(k_zero, dim3(1024), dim3(256), 0, s, b->d_Gt.p, b->gt_total);
    auto class_launch = [&](const qf_engine::Launch& L, hipStream_t stream) -> int {
        qf::LaunchTo q(stream);
        if (L.tile == 2) {
            qf::FockCoopLaunch fc = qf::fock_coop_launcher(L.cb, L.ck);
            if (!fc) return fail(QF_ERR_ARG, "no wave-per-quartet kernel for class");
            fc(b->d_tasks.p + L.offset, L.count, b->d_blocks.p, b->d_moldesc.p, 0, b->persist, b->d_cscratch.p + L.gslot, q);
        } else if (L.tile) {
            qf::FockTileLaunch ft = qf::fock_tile_launcher(L.cb, L.ck);
            if (!ft) return fail(QF_ERR_ARG, "no tile kernel for class");
            ft(b->d_groups.p + L.goffset, L.gcount, b->d_tasks.p, b->d_blocks.p, b->d_moldesc.p, L.fp32, 0, L.waves,
               L.lds, b->persist, q);
        } else {
            qf::FockLaunch f = qf::fock_launcher(L.cb, L.ck);
            if (!f) return fail(QF_ERR_ARG, "no per-lane kernel for class");
            if (f(b->d_tasks.p + L.offset, L.count, b->d_blocks.p, b->d_moldesc.p, L.fp32, 0, b->persist, q))
                return fail(QF_ERR_ARG, kDirectFp32Refused);
        }
        return QF_OK;
    };
    if (b->timing) {
        for (size_t li = 0; li < b->launches.size(); ++li) {
            while (b->ev_pool.size() < b->ev_used + 2) {
                hipEvent_t ev;
                QF_HIP(hipEventCreate(&ev));
                b->ev_pool.push_back(ev);
            }
            hipEvent_t ea = b->ev_pool[b->ev_used], eb = b->ev_pool[b->ev_used + 1];
            b->ev_used += 2;
            b->ev_launch.push_back((int)li);
            QF_HIP(hipEventRecord(ea, s));
            const int rc = class_launch(b->launches[li], s);
            if (rc) return rc;
            QF_HIP(hipEventRecord(eb, s));
        }
    } else {
        const int rc = issue_forked(b->order.size() > 1 ? b->side : nullptr, s, b->order,
                                    [&](int li, hipStream_t q) { return class_launch(b->launches[li], q); });
        if (rc) return rc;
    }
    hipLaunchKernelGGL(k_finalize_batch, dim3((b->max_n2 + 255) / 256, nm), dim3(256), 0, s, b->d_bm.p,
                       b->replicas);
    QF_HIP(hipGetLastError());
    return QF_OK;
}

}  // namespace

extern "C" {

int qf_batch_create_ext(qf_engine* const* engines, int count, int replicas, const double* const* d_P,
                        double* const* d_F, qf_batch** out)
{
    if (!engines || count <= 0 || !out) return fail(QF_ERR_ARG, "engines/count/out");
    if ((d_P == nullptr) != (d_F == nullptr)) return fail(QF_ERR_ARG, "give both d_P and d_F or neither");
    if (replicas < 1 || replicas > 64) return fail(QF_ERR_ARG, "replicas must be in 1..64");
    *out = nullptr;
    auto* b = new qf_batch();
    b->device = engines[0]->device;
    b->replicas = replicas;
    b->persist = engines[0]->persist;
    int rc = QF_OK;
    auto bail = [&](int code) {
        delete b;
        return code;
    };
    if (hipSetDevice(b->device) != hipSuccess) return bail(fail(QF_ERR_BADDEVICE, "hipSetDevice"));
    for (int i = 0; i < count; ++i) {
        qf_engine* e = engines[i];
        if (!e) return bail(fail(QF_ERR_ARG, "NULL engine"));
        if (e->device != b->device) return bail(fail(QF_ERR_ARG, "engines of a batch must share one device"));
        rc = prepare(e);
        if (rc) return bail(rc);
        b->engs.push_back(e);
        b->gens.push_back(e->generation);
    }
    // pooled buffers
    size_t np = 0, ncm = 0;
    std::vector<size_t> poff, cmoff, gtoff;
    for (qf_engine* e : b->engs) {
        const size_t n2 = (size_t)e->nbasis * e->nbasis;
        poff.push_back(np);
        cmoff.push_back(ncm);
        gtoff.push_back(b->gt_total);
        np += n2;
        ncm += (size_t)e->nshell * e->nshell;
        b->gt_total += n2 * replicas;
        b->max_n2 = std::max<int>(b->max_n2, (int)n2);
        b->max_ns2 = std::max<int>(b->max_ns2, e->nshell * e->nshell);
    }
    if ((!d_P && (b->d_P.resize(np) != hipSuccess || b->d_F.resize(np) != hipSuccess)) || b->d_Gs.resize(np) != hipSuccess || b->d_cm.resize(ncm) != hipSuccess ||
        b->d_Gt.resize(b->gt_total) != hipSuccess)
        return bail(fail(QF_ERR_MEMORY, "batch buffers"));
    if (!d_P && (hipMemset(b->d_P.p, 0, np * sizeof(double)) != hipSuccess ||
                 hipMemset(b->d_F.p, 0, np * sizeof(double)) != hipSuccess))
        return bail(fail(QF_ERR_HIP, "hipMemset"));
    // combined tables
    std::vector<qf::PairBlock> blocks;
    std::vector<qf::MolDesc> md;
    std::vector<int> boff;
    for (int i = 0; i < count; ++i) {
        qf_engine* e = b->engs[i];
        boff.push_back((int)blocks.size());
        for (qf::PairBlock pb : e->hblocks) {
            pb.mol = i;
            blocks.push_back(pb);
        }
        if (d_P && (!d_P[i] || !d_F[i])) return bail(fail(QF_ERR_ARG, "NULL density/Fock pointer"));
        qf::MolDesc m{};
        m.P = d_P ? d_P[i] : b->d_P.p + poff[i];
        m.PJ = m.P;
        m.G = b->d_Gt.p + gtoff[i];
        m.cutmat = b->d_cm.p + cmoff[i];
        m.nbasis = e->nbasis;
        m.nshell = e->nshell;
        m.cutoff = e->cutoff;
        m.primlim = e->primlim;
        m.hyb = e->hyb;
        m.replicas = replicas;
        m.split = (e->prec == QF_PREC_MIXED) ? e->split_thr : 0.0;
        md.push_back(m);
        BatchMol bm{};
        bm.P = m.P;
        bm.F = d_F ? d_F[i] : b->d_F.p + poff[i];
        bm.Gt = m.G;
        bm.Gs = b->d_Gs.p + poff[i];
        bm.cm = b->d_cm.p + cmoff[i];
        bm.f0 = e->shell_f0();
        bm.f1 = e->shell_f1();
        bm.n = e->nbasis;
        bm.ns = e->nshell;
        b->mols.push_back(bm);
    }
    std::vector<qf::Task> tasks;
    std::vector<qf::TileGroup> groups;
    // The molecules of a batch fill the GPU together, so their launch shapes are
    // those of the one molecule with as much work: quartets grow about as the
    // cube of the functions.  (With each molecule's own shapes, primitive pieces
    // of one pair and four tasks a workgroup for the small ones, 48 molecules of
    // 19-156 functions took 24.7 ms a build, with these 16.0.)
    double cube = 0.0;
    for (const qf_engine* e : b->engs) cube += std::pow((double)e->nbasis, 3.0);
    const int size = (int)std::cbrt(cube);
    std::vector<ClassShape> shapes(count);
    TaskScratch sc;
    // room for the usual number (pieces and windows differ from the engines' own):
    // growing would touch every page twice, what is not used is never touched
    size_t expect = 0;
    for (const qf_engine* e : b->engs) expect += e->tasks.size();
    tasks.reserve(4 * expect);
    groups.reserve(4 * expect);
    for (int cb = 0; cb < kNPC; ++cb)
        for (int ck = 0; ck <= cb; ++ck)
            for (int fp32 = 0; fp32 < 2; ++fp32)
                for (int tile = 0; tile < 3; ++tile) {
                    if (tile == 0)
                        for (int i = 0; i < count; ++i)
                            if ((rc = class_shape(b->engs[i], cb, ck, fp32, size, false, shapes[i]))) return bail(rc);
                    qf_engine::Launch C{};
                    C.cb = cb;
                    C.ck = ck;
                    C.fp32 = fp32;
                    C.tile = tile;
                    C.offset = (int)tasks.size();
                    C.goffset = (int)groups.size();
                    C.waves = 1;
                    for (int i = 0; i < count; ++i) {
                        if (!shapes[i].runs || shapes[i].kind != tile) continue;
                        qf_engine::Launch L;
                        if ((rc = class_tasks(b->engs[i], cb, ck, fp32, shapes[i], boff[i], sc, tasks, groups, nullptr,
                                              false, L)))
                            return bail(rc);
                        C.lds = std::max(C.lds, L.lds);
                        C.waves = std::max(C.waves, L.waves);
                    }
                    C.count = (int)tasks.size() - C.offset;
                    C.gcount = (int)groups.size() - C.goffset;
                    if (C.count == 0) continue;
                    if (tile == 1)
                        longest_first(groups, C.goffset, tasks);
                    else
                        longest_first(tasks, C.offset);
                    b->launches.push_back(C);
                }
    const size_t gdoubles = place_slots(b->launches);
    if (gdoubles && b->d_cscratch.resize(gdoubles) != hipSuccess)
        return bail(fail(QF_ERR_MEMORY, "batch global slot buffer"));
    if (b->d_blocks.upload(blocks) != hipSuccess || b->d_tasks.upload(tasks) != hipSuccess ||
        b->d_groups.upload(groups) != hipSuccess || b->d_moldesc.upload(md) != hipSuccess ||
        b->d_bm.upload(b->mols) != hipSuccess)
        return bail(fail(QF_ERR_HIP, "batch table upload"));
    qf_engine::Plan order;
    stream_order(b->launches, tasks, order);
    b->order = std::move(order.order);
    b->side = SidePool::get().take(b->device);   // null: the batch runs on the caller's stream alone
    *out = b;
    return QF_OK;
}

int qf_batch_create(qf_engine* const* engines, int count, int replicas, qf_batch** out)
{
    return qf_batch_create_ext(engines, count, replicas, nullptr, nullptr, out);
}

void qf_batch_destroy(qf_batch* b)
{
    if (!b) return;
    (void)hipSetDevice(b->device);
    delete b;
}

int qf_batch_size(qf_batch* b) { return b ? (int)b->mols.size() : -1; }

double* qf_batch_density(qf_batch* b, int i)
{
    if (!b || i < 0 || i >= (int)b->mols.size()) return nullptr;
    return const_cast<double*>(b->mols[i].P);
}

double* qf_batch_fock(qf_batch* b, int i)
{
    if (!b || i < 0 || i >= (int)b->mols.size()) return nullptr;
    return b->mols[i].F;
}

const double* qf_batch_g(qf_batch* b, int i)
{
    if (!b || i < 0 || i >= (int)b->mols.size()) return nullptr;
    return b->mols[i].Gs;
}

int qf_batch_set_graph(qf_batch* b, int enable)
{
    if (!b) return fail(QF_ERR_ARG, "NULL");
    b->use_graph = enable != 0;
    return QF_OK;
}

int qf_batch_build(qf_batch* b, void* stream)
{
    if (!b) return fail(QF_ERR_ARG, "NULL");
    // the batch (and its graph) holds pointers into every engine's pair and
    // task tables: a re-prepared engine has replaced them
    for (size_t i = 0; i < b->engs.size(); ++i)
        if (b->engs[i]->generation != b->gens[i] || !b->engs[i]->prepared)
            return fail(QF_ERR_STATE, "engine " + std::to_string(i) +
                                          " was changed or re-prepared after the batch was created; create the batch again");
    QF_HIP(hipSetDevice(b->device));
    hipStream_t s = (hipStream_t)stream;
    if (!b->use_graph || b->timing) return batch_issue(b, s);
    if (!b->exec) {
        // capture on a private stream (capture needs a non-legacy stream)
        if (!b->cap_stream) QF_HIP(hipStreamCreateWithFlags(&b->cap_stream, hipStreamNonBlocking));
        QF_HIP(hipStreamBeginCapture(b->cap_stream, hipStreamCaptureModeThreadLocal));
        int rc = batch_issue(b, b->cap_stream);
        hipGraph_t g = nullptr;
        hipError_t ce = hipStreamEndCapture(b->cap_stream, &g);
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (ce != hipSuccess) return fail(QF_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(ce));
        b->graph = g;
        QF_HIP(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
    }
    QF_HIP(hipGraphLaunch(b->exec, s));
    return QF_OK;
}

int qf_fock_build_batch(qf_engine* const* engines, int count, const double* const* d_P, double* const* d_F,
                        void* stream)
{
    // One-shot form of the batch API: a temporary batch, one launch per
    // class for all engines.  Repeated builds should keep a qf_batch.
    if (!engines || !d_P || count <= 0) return fail(QF_ERR_ARG, "NULL");
    qf_batch* b = nullptr;
    int rc = qf_batch_create(engines, count, 2, &b);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    for (int i = 0; i < count && !rc; ++i) {
        const size_t n2 = (size_t)b->mols[i].n * b->mols[i].n;
        if (hipMemcpyAsync(const_cast<double*>(b->mols[i].P), d_P[i], n2 * sizeof(double), hipMemcpyDeviceToDevice,
                           s) != hipSuccess)
            rc = fail(QF_ERR_HIP, "hipMemcpyAsync (batch density)");
    }
    if (!rc) rc = batch_issue(b, s);
    for (int i = 0; i < count && !rc; ++i) {
        const int n2 = b->mols[i].n * b->mols[i].n;
        if (d_F && d_F[i])
            hipLaunchKernelGGL(k_add, dim3((n2 + 255) / 256), dim3(256), 0, s, d_F[i], b->mols[i].Gs, n2);
        if (hipMemcpyAsync(engines[i]->d_Gs.p, b->mols[i].Gs, (size_t)n2 * sizeof(double), hipMemcpyDeviceToDevice,
                           s) != hipSuccess)
            rc = fail(QF_ERR_HIP, "hipMemcpyAsync (batch G)");
    }
    if (!rc && hipStreamSynchronize(s) != hipSuccess) rc = fail(QF_ERR_HIP, "hipStreamSynchronize");
    qf_batch_destroy(b);
    return rc;
}

int qf_batch_set_density_host(qf_batch* b, int i, const double* P)
{
    if (!b || !P || i < 0 || i >= (int)b->mols.size()) return fail(QF_ERR_ARG, "batch density");
    QF_HIP(hipSetDevice(b->device));
    const size_t n2 = (size_t)b->mols[i].n * b->mols[i].n;
    QF_HIP(hipMemcpy(const_cast<double*>(b->mols[i].P), P, n2 * sizeof(double), hipMemcpyHostToDevice));
    return QF_OK;
}

int qf_batch_get_host(qf_batch* b, int i, double* G, double* F)
{
    if (!b || i < 0 || i >= (int)b->mols.size()) return fail(QF_ERR_ARG, "batch index");
    QF_HIP(hipSetDevice(b->device));
    const size_t n2 = (size_t)b->mols[i].n * b->mols[i].n;
    if (G) QF_HIP(hipMemcpy(G, b->mols[i].Gs, n2 * sizeof(double), hipMemcpyDeviceToHost));
    if (F) QF_HIP(hipMemcpy(F, b->mols[i].F, n2 * sizeof(double), hipMemcpyDeviceToHost));
    return QF_OK;
}

int qf_batch_clear_fock(qf_batch* b, void* stream)
{
    if (!b) return fail(QF_ERR_ARG, "NULL");
    QF_HIP(hipSetDevice(b->device));
    hipLaunchKernelGGL(k_clear_batch, dim3((b->max_n2 + 255) / 256, (unsigned)b->mols.size()), dim3(256), 0,
                       (hipStream_t)stream, b->d_bm.p);
    QF_HIP(hipGetLastError());
    return QF_OK;
}

int qf_batch_launch_count(qf_batch* b) { return b ? (int)b->launches.size() : -1; }

int qf_batch_launch_info(qf_batch* b, int idx, int* cb, int* ck, int* fp32, int* ntasks)
{
    if (!b || idx < 0 || idx >= (int)b->launches.size()) return fail(QF_ERR_ARG, "launch index");
    const auto& L = b->launches[idx];
    *cb = L.cb;
    *ck = L.ck;
    *fp32 = L.fp32;
    *ntasks = L.count;
    return QF_OK;
}

int qf_batch_set_timing(qf_batch* b, int enable)
{
    if (!b) return fail(QF_ERR_ARG, "NULL");
    b->timing = enable != 0;
    b->ev_used = 0;
    b->ev_launch.clear();
    return QF_OK;
}

int qf_batch_read_timing(qf_batch* b, double* ms_per_launch, int* calls_per_launch)
{
    if (!b) return fail(QF_ERR_ARG, "NULL");
    const size_t nl = b->launches.size();
    for (size_t k = 0; k < nl; ++k) {
        ms_per_launch[k] = 0.0;
        calls_per_launch[k] = 0;
    }
    if (b->ev_used) QF_HIP(hipEventSynchronize(b->ev_pool[b->ev_used - 1]));
    for (size_t r = 0; r < b->ev_launch.size(); ++r) {
        if (b->ev_launch[r] < 0 || (size_t)b->ev_launch[r] >= nl) continue;
        float ms = 0.0f;
        QF_HIP(hipEventElapsedTime(&ms, b->ev_pool[2 * r], b->ev_pool[2 * r + 1]));
        ms_per_launch[b->ev_launch[r]] += ms;
        calls_per_launch[b->ev_launch[r]] += 1;
    }
    b->ev_used = 0;
    b->ev_launch.clear();
    return QF_OK;
}

}  // extern "C"
