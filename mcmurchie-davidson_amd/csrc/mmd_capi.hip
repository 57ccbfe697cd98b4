// libmmd host runtime: the C ABI declared in include/mmd.h.
//
// A context owns one HIP stream, the Boys table, the basis (per function and
// per shell), shell-pair / primitive-pair tables, Schwarz data, the density
// and Fock scratch buffers and the per-class survivor lists.  Callers own
// every input and output pointer.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdarg.h>
#include <stddef.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/mmd.h"
#include <rocblas/rocblas.h>
#include "mmd_batch.h"
#include "mmd_device.h"
#include "mmd_gemm.h"
#include "mmd_grad.h"
#include "mmd_kernels.h"
#include "mmd_hostcopy.h"
#include "mmd_pairs.h"
#include "mmd_pool.h"
#include "mmd_scf.h"
#include "mmd_types.h"

using namespace mmd;

namespace mmd {
std::recursive_mutex& device_alloc_mutex()
{
    static std::recursive_mutex mu;
    return mu;
}
}  // namespace mmd

namespace {

thread_local std::string g_last_error;

int fail(int code, const char* fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

#define HIP_TRY(expr)                                                                           \
    do {                                                                                        \
        hipError_t e_ = (expr);                                                                 \
        if (e_ != hipSuccess) {                                                                 \
            if (e_ == hipErrorOutOfMemory) return fail(MMD_ERR_NOMEM, "%s: %s", #expr, hipGetErrorString(e_)); \
            return fail(MMD_ERR_DEVICE, "%s: %s", #expr, hipGetErrorString(e_));                \
        }                                                                                       \
    } while (0)

struct Shell {
    int l, np, p0, bf0;
    int mol;   // molecule of the shell's functions
    double x, y, z;
};

template <class T>
struct DevBuf {
    T* p = nullptr;
    size_t n = 0;
    ~DevBuf() { release(); }
    void release()
    {
        if (p) {
            std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
            (void)hipFree(p);
        }
        p = nullptr;
        n = 0;
    }
    hipError_t reserve(size_t count)
    {
        if (count <= n && p) return hipSuccess;
        std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
        release();
        if (count == 0) count = 1;
        hipError_t e = device_malloc((void**)&p, count * sizeof(T));
        if (e == hipSuccess) n = count;
        return e;
    }
};

}  // namespace

// ---------------------------------------------------------------------------
// Static scratch of mmd_fock_delta_noalloc: one array per device (each GPU
// the library runs on holds its own copy until the process ends).  Host code
// never passes the array's name to a kernel (on the host it is a stand-in,
// not a device address): every use goes through the address that
// hipGetSymbolAddress returned for the device, looked up once per device when
// the first context on it is created (scratch_for_device).
// ---------------------------------------------------------------------------
constexpr size_t NOALLOC_SCRATCH_BYTES = size_t(16) << 20;   // 16 MiB
constexpr int NPRIM_SLOTS = 4 * NQCLASS;   // survivor counters of one Fock build
// A build's counters, in one block: what the host reads back (survivors, list
// lengths) first, then the row kernels' unit counters.
struct FockCounters {
    unsigned long long nprim[NPRIM_SLOTS];   // see FockScratch::nprim
    int count[2 * NQCLASS];                  // survivor-list lengths (FP64 lists, then FP32)
    int nlive[NQCLASS];                      // live units of a batch's classes
    int pad[ROW_QUEUE_PAD];
    int rowctr[2 * NQCLASS][ROW_QUEUES * ROW_QUEUE_PAD];   // unit queues, FP64 then FP32 pass
};
constexpr int FOCK_COUNTER_WORDS = (int)(sizeof(FockCounters) / sizeof(int));
constexpr int FOCK_REPORT_WORDS = (int)(offsetof(FockCounters, nlive) / sizeof(int));

// Per-class sums over profiled builds; index 0 the FP64 launches, 1 the FP32 tier.
struct ProfileSum {
    int64_t nquart[2] = {0, 0}, nprim[2] = {0, 0};
    double ms[2] = {0.0, 0.0};
    int64_t builds = 0;
};
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[MAX_DEVICES] = {};

// Device address of `scratch` on the current device (device_id), looked up
// on the first call for that device.
int scratch_for_device(int device_id, void** out)
{
    if (device_id < 0 || device_id >= MAX_DEVICES) return fail(MMD_ERR_ARG, "device id out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[device_id]) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return fail(MMD_ERR_DEVICE, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        g_scratch_ptr[device_id] = ptr;
    }
    *out = g_scratch_ptr[device_id];
    return MMD_OK;
}
}  // namespace

struct mmd_ctx {
    int device = 0;
    void* noalloc_scratch = nullptr;    // this device's `scratch` (device address)
    hipStream_t st = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // side streams for concurrent class kernels (default priority), with the
    // fork / join events that order them against st
    static constexpr int NSIDE = 7;
    hipStream_t side[NSIDE] = {};
    hipEvent_t evfork = nullptr, evjoin[NSIDE] = {};
    int nstreams = 1 + NSIDE;           // streams the Fock classes are spread over
    double last_fock_ms = 0.0;
    int64_t last_nsurv = 0, last_nsurv_fp32 = 0;   // shell quartets of the last symmetrised build
    double fp32_below = 0.0;                        // FP32 tier: quartets with bound below this (0: off)
    DevBuf<float> d_boysf;

    // basis, per function
    int nbf = 0;
    std::vector<BFDesc> bf;
    std::vector<double> bf_exp, bf_w;
    DevBuf<BFDesc> d_bf;
    DevBuf<double> d_bf_exp, d_bf_w;
    DevBuf<double> d_boys;

    // basis, per shell
    bool shells_ok = false;
    std::string shells_err;
    std::vector<Shell> shells;
    std::vector<double> sh_exp, sh_w, gcomp;
    DevBuf<double> d_gcomp;
    DevBuf<int> d_sh_bf0, d_sh_nbf;
    DevBuf<OneeShell> d_oshell;         // shells for the one-electron kernels
    DevBuf<double> d_sh_exp, d_sh_w;
    DevBuf<int2> d_onee_list;           // every shell pair of each molecule, by pair class
    int onee_off[NPAIRCLASS + 1] = {0};
    bool onee_list_ok = false;

    // shell pairs (grouped by pair class, sorted inside each class)
    bool pairs_ok = false;
    int pc_off[NPAIRCLASS + 1] = {0};
    int pc_npp[NPAIRCLASS] = {0}, pc_maxpp[NPAIRCLASS] = {0};   // primitive pairs of a class, largest count of a pair
    DevBuf<int2> d_ranges;              // per class and molecule: its pairs {first, end} in the class
    std::vector<int2> pair_ranges;      // and on the host, with the bra slices if no primitive pair is
    std::vector<int64_t> pair_slices;   // screened out, and the primitive pairs of each class
    int64_t pair_prims[NPAIRCLASS] = {0};
    DevBuf<int> w_count, w_entry, w_scan, w_ints;   // work of the table build (PairWork)
    DevBuf<double> w_q;
    DevBuf<uint16_t> w_keep;
    DevBuf<ShellPair> d_pairs;
    DevBuf<PrimPair> d_pp;
    DevBuf<KetScreen> d_kscr;    // ket tables of the row kernels
    DevBuf<KetRef> d_kref;
    DevBuf<double> d_kpp;
    int64_t kpp_stride = 0;
    DevBuf<double> jk_mats;      // N x N matrices of the tensor calls
    DevBuf<double> d_onee;   // S, T, V, M (3), L (3) of mmd_one_electron
    DevBuf<double> d_ns;     // overlap powers: S, X, U and the Newton-Schulz work (8 N^2 + 2)

    // Schwarz
    bool schwarz_ok = false;
    DevBuf<double> d_schwarz, d_sqS;

    // quartet classes
    int64_t qc_total[NQCLASS] = {0};
    int64_t qc_off[NQCLASS + 1] = {0};
    DevBuf<int2> d_surv;
    DevBuf<FockCounters> d_ctr;
    FockCounters* h_ctr = nullptr;   // pinned: the counters of the last build
    int* h_pairs = nullptr;          // and the table build's report, after them

    // atoms
    int natom = 0;
    DevBuf<double> d_atoms;
    DevBuf<double> g_PW;                // gradient: P, W and the natom x 3 result
    DevBuf<int> g_atom;                 // gradient: atom of each basis function
    double last_grad_ms = 0.0;
    // gradient by shell class: exponent of the first function of every
    // primitive pair, the classes' bra slices (of grad_pslice primitive pairs,
    // and of one for the workgroup-per-primitive-quartet kernels) and flat primitive-pair lists,
    // made from the pair table on first use
    DevBuf<double> d_ppa, g_rep;
    DevBuf<int4> g_slices;
    DevBuf<int2> g_flat;
    int g_slice_off[NPAIRCLASS + 1] = {0}, g_one_off[NPAIRCLASS + 1] = {0}, g_flat_off[NPAIRCLASS + 1] = {0};
    bool grad_plan_ok = false;

    // integral-block kernels: staged bra data per pair class (made from the
    // pair table on first use), copies of the raw G
    DevBuf<double> d_btab, d_graw, d_qraw;
    size_t btab_off[NPAIRCLASS] = {0};
    bool btab_ok = false, qraw_ok = false;

    // Molecules of a block-diagonal basis (mmd_set_molecules; one molecule
    // unless set): molecule m owns functions [mol_f0[m], mol_f0[m] + mol_n[m])
    // and shells [mol_s0[m], mol_s0[m + 1]); pairs and quartets never mix
    // molecules.  rw: the largest molecule (width of the class kernels' LDS
    // rows); plist: the same-molecule function pairs p >= q.
    int nmol = 1;
    std::vector<int> mol_f0{0}, mol_n{0}, mol_s0{0, 0};
    std::vector<int2> mol_atoms;        // per molecule: first atom, number of atoms
    DevBuf<int2> d_mol_atoms;
    DevBuf<int2> d_plist;
    DevBuf<int4> d_mol_blocks;          // per molecule: first function, functions, shells [s0, s1)
    DevBuf<double> d_mol_dmax;          // per molecule: max |dP| of the build
    int64_t npl = 0;
    int rw = 0;

    // density / Fock scratch
    DevBuf<double> d_D, d_Dim, d_absD, d_Dsh, d_G, d_Gout;

    // per-class statistics of the last symmetrised Fock build
    int profiling = 0;                  // 0 off; 1 events, classes concurrent; 2 events, classes serial
    hipEvent_t evc[3 * NQCLASS] = {};   // per class: start, after the FP64 launch, end
    // Stream plan of the Fock build: class durations measured with the
    // per-class events in one build out of PLAN_EVERY (0: not measured yet).
    static constexpr int PLAN_EVERY = 16;
    double plan_ms[NQCLASS] = {0};
    int plan_countdown = 0;
    bool plan_measuring = false;
    // The six classes with both a row kernel and a matrix-core kernel:
    // impl_mode 0 takes the row kernels, 1 the matrix cores, 2 times both on
    // the first two measured builds of a pair table (the classes running side
    // by side as usual) and keeps the faster per class (impl_choice: -1
    // undecided, 0 row, 1 matrix cores).
    int impl_mode = 2;
    int impl_choice[NQCLASS];
    int ket_slice[NQCLASS];             // mmd_set_ket_slices (KSLICE_DEFAULT until set)
    int tune_phase = 0;
    double tune_ms[2][NQCLASS] = {};
    bool tune_measuring = false;
    // Work units of the row-kernel classes (built once per pair table):
    // class qc owns units [unit_off[qc], unit_off[qc+1]).
    DevBuf<int4> d_units;
    DevBuf<UnitBound> d_ubound;         // per unit, in the same order
    DevBuf<int> d_live;
    int64_t unit_off[NQCLASS + 1] = {0};
    bool units_ok = false;
    size_t max_lds = 65536;             // LDS a class launch may use (mmd_set_lds_limit)
    size_t max_lds_device = 65536;      // the device's limit per workgroup
    size_t lds_per_block = 65536;       // the device's LDS limit per workgroup, as reported
    bool last_row_kernel[NQCLASS] = {};
    int64_t st_nquart[NQCLASS] = {0};

    // batched RHF (mmd_batch_rhf): N x N block-diagonal matrices, per-molecule
    // work, DIIS windows and state
    DevBuf<double> b_H, b_X, b_U, b_F, b_P, b_Pold, b_dP, b_G, b_work, b_diis, b_mo;
    DevBuf<BatchMol> b_mol;
    DevBuf<BatchState> b_state;
    DevBuf<int> b_flag, b_count;

    // GPU-resident SCF loop (mmd_scf_*): matrices, DIIS window, BLAS handle
    rocblas_handle blas = nullptr;
    int scf_n = 0, scf_nocc = 0;
    DevBuf<double> s_H, s_S, s_X, s_F, s_P, s_Pold, s_G, s_dP, s_T1, s_T2, s_C, s_stats, s_dots;
    DevBuf<double> s_Fset, s_Eset;   // DIIS window: 8 slots of N*N each
    std::vector<int> s_order;        // slots of the window, oldest first
    std::vector<double> s_B;         // 8 x 8 error overlaps, window order
    int64_t st_nprim[NQCLASS] = {0};
    double st_ms[NQCLASS] = {0};
    ProfileSum psum[NQCLASS];           // sums over the builds since profiling was turned on
};

namespace {

int check_ctx(mmd_ctx* ctx)
{
    if (!ctx) return fail(MMD_ERR_ARG, "null context");
    hipError_t e = hipSetDevice(ctx->device);
    if (e != hipSuccess) return fail(MMD_ERR_DEVICE, "hipSetDevice: %s", hipGetErrorString(e));
    return MMD_OK;
}

// Group consecutive basis functions into complete Cartesian shells in the
// reference's component order with a common centre and exponents and
// weights that differ by a per-component factor only.
void build_shells(mmd_ctx* c)
{
    c->shells.clear();
    c->sh_exp.clear();
    c->sh_w.clear();
    c->gcomp.assign(c->nbf, 1.0);
    c->shells_ok = false;
    int i = 0;
    while (i < c->nbf) {
        const BFDesc& b0 = c->bf[i];
        const int L = b0.l + b0.m + b0.n;
        const int nc = ncart(L);
        if (b0.l != L || i + nc > c->nbf) {
            c->shells_err = "basis functions do not form complete Cartesian shells";
            return;
        }
        for (int k = 0; k < nc; ++k) {
            const BFDesc& bk = c->bf[i + k];
            bool ok = bk.l == comp_lx(L, k) && bk.m == comp_ly(L, k) && bk.n == comp_lz(L, k) && bk.np == b0.np
                   && bk.x == b0.x && bk.y == b0.y && bk.z == b0.z;
            if (ok) {
                const double g = c->bf_w[bk.p0] / c->bf_w[b0.p0];
                for (int p = 0; p < b0.np && ok; ++p) {
                    ok = c->bf_exp[bk.p0 + p] == c->bf_exp[b0.p0 + p];
                    const double gp = c->bf_w[bk.p0 + p] / c->bf_w[b0.p0 + p];
                    ok = ok && fabs(gp - g) <= 1e-12 * fabs(g);
                }
                c->gcomp[i + k] = g;
            }
            if (!ok) {
                c->shells_err = "basis functions do not form complete Cartesian shells";
                return;
            }
        }
        Shell s;
        s.l = L;
        s.mol = b0.pad;
        s.np = b0.np;
        s.p0 = (int)c->sh_exp.size();
        s.bf0 = i;
        s.x = b0.x;
        s.y = b0.y;
        s.z = b0.z;
        for (int p = 0; p < b0.np; ++p) {
            c->sh_exp.push_back(c->bf_exp[b0.p0 + p]);
            c->sh_w.push_back(c->bf_w[b0.p0 + p]);
        }
        c->shells.push_back(s);
        i += nc;
    }
    c->shells_ok = true;
}

int upload_shells(mmd_ctx* c)
{
    HIP_TRY(c->d_gcomp.reserve(c->nbf));
    HIP_TRY(hipMemcpyAsync(c->d_gcomp.p, c->gcomp.data(), sizeof(double) * c->nbf, hipMemcpyHostToDevice, c->st));
    const int ns = (int)c->shells.size();
    std::vector<int> b0(ns), nb(ns);
    for (int s = 0; s < ns; ++s) {
        b0[s] = c->shells[s].bf0;
        nb[s] = ncart(c->shells[s].l);
    }
    HIP_TRY(c->d_sh_bf0.reserve(ns));
    HIP_TRY(c->d_sh_nbf.reserve(ns));
    HIP_TRY(hipMemcpyAsync(c->d_sh_bf0.p, b0.data(), sizeof(int) * ns, hipMemcpyHostToDevice, c->st));
    HIP_TRY(hipMemcpyAsync(c->d_sh_nbf.p, nb.data(), sizeof(int) * ns, hipMemcpyHostToDevice, c->st));
    std::vector<OneeShell> os(std::max(ns, 1));
    for (int k = 0; k < ns; ++k) {
        const Shell& sh = c->shells[k];
        os[k] = OneeShell{sh.x, sh.y, sh.z, sh.l, sh.np, sh.p0, sh.bf0, sh.mol, 0};
    }
    HIP_TRY(c->d_oshell.reserve(os.size()));
    HIP_TRY(c->d_sh_exp.reserve(c->sh_exp.size()));
    HIP_TRY(c->d_sh_w.reserve(c->sh_w.size()));
    HIP_TRY(hipMemcpyAsync(c->d_oshell.p, os.data(), sizeof(OneeShell) * os.size(), hipMemcpyHostToDevice, c->st));
    HIP_TRY(hipMemcpyAsync(c->d_sh_exp.p, c->sh_exp.data(), sizeof(double) * c->sh_exp.size(), hipMemcpyHostToDevice,
                           c->st));
    HIP_TRY(hipMemcpyAsync(c->d_sh_w.p, c->sh_w.data(), sizeof(double) * c->sh_w.size(), hipMemcpyHostToDevice,
                           c->st));
    HIP_TRY(hipStreamSynchronize(c->st));
    c->onee_list_ok = false;
    return MMD_OK;
}

// Shells [mol_s0[m], mol_s0[m+1]) of each molecule (shells never span two),
// and, for a batch, the molecules' blocks {f0, n, s0, s1} on the device.
int molecule_shell_ranges(mmd_ctx* c)
{
    const int ns = (int)c->shells.size();
    c->mol_s0.assign(c->nmol + 1, ns);
    for (int I = ns - 1; I >= 0; --I) c->mol_s0[c->shells[I].mol] = I;
    for (int m = c->nmol - 1; m >= 0; --m)
        if (c->mol_s0[m] > c->mol_s0[m + 1]) c->mol_s0[m] = c->mol_s0[m + 1];
    if (c->nmol > 1) {
        std::vector<int4> blk(c->nmol);
        for (int m = 0; m < c->nmol; ++m)
            blk[m] = make_int4(c->mol_f0[m], c->mol_n[m], c->mol_s0[m], c->mol_s0[m + 1]);
        HIP_TRY(c->d_mol_blocks.reserve(c->nmol));
        HIP_TRY(c->d_mol_dmax.reserve(c->nmol));
        HIP_TRY(hipMemcpyAsync(c->d_mol_blocks.p, blk.data(), sizeof(int4) * c->nmol, hipMemcpyHostToDevice, c->st));
    }
    return MMD_OK;
}

// Every shell pair of each molecule (l_a >= l_b), grouped by pair class,
// for the shell-pair one-electron and Schwarz kernels; built once per basis.
int onee_pair_list(mmd_ctx* c)
{
    if (c->onee_list_ok) return MMD_OK;
    if (int rc = molecule_shell_ranges(c)) return rc;
    std::vector<std::vector<int2>> byclass(NPAIRCLASS);
    std::vector<int2>& ranges = c->pair_ranges;
    ranges.assign((size_t)NPAIRCLASS * c->nmol, make_int2(0, 0));
    c->pair_slices.assign((size_t)NPAIRCLASS * c->nmol, 0);
    for (int64_t& p : c->pair_prims) p = 0;
    for (int m = 0; m < c->nmol; ++m) {
        for (int pc = 0; pc < NPAIRCLASS; ++pc) ranges[(size_t)pc * c->nmol + m].x = (int)byclass[pc].size();
        for (int I = c->mol_s0[m]; I < c->mol_s0[m + 1]; ++I)
            for (int J = c->mol_s0[m]; J <= I; ++J) {
                int a = I, b = J;
                if (c->shells[I].l < c->shells[J].l) std::swap(a, b);
                const int pc = pair_class(c->shells[a].l, c->shells[b].l), np = c->shells[a].np * c->shells[b].np;
                byclass[pc].push_back(make_int2(a, b));
                c->pair_prims[pc] += np;
                c->pair_slices[(size_t)pc * c->nmol + m] += (np + PSLICE - 1) / PSLICE;
            }
        for (int pc = 0; pc < NPAIRCLASS; ++pc) ranges[(size_t)pc * c->nmol + m].y = (int)byclass[pc].size();
    }
    HIP_TRY(c->d_ranges.reserve(ranges.size()));
    HIP_TRY(hipMemcpyAsync(c->d_ranges.p, ranges.data(), sizeof(int2) * ranges.size(), hipMemcpyHostToDevice, c->st));
    std::vector<int2> all;
    for (int pc = 0; pc < NPAIRCLASS; ++pc) {
        c->onee_off[pc] = (int)all.size();
        all.insert(all.end(), byclass[pc].begin(), byclass[pc].end());
    }
    c->onee_off[NPAIRCLASS] = (int)all.size();
    HIP_TRY(c->d_onee_list.reserve(std::max<size_t>(all.size(), 1)));
    HIP_TRY(hipMemcpyAsync(c->d_onee_list.p, all.data(), sizeof(int2) * all.size(), hipMemcpyHostToDevice, c->st));
    HIP_TRY(hipStreamSynchronize(c->st));
    c->onee_list_ok = true;
    return MMD_OK;
}

OneeArgs onee_args(const mmd_ctx* c)
{
    OneeArgs A{};
    A.shells = c->d_oshell.p;
    A.exps = c->d_sh_exp.p;
    A.wts = c->d_sh_w.p;
    A.gcomp = c->d_gcomp.p;
    A.atoms = c->natom ? c->d_atoms.p : nullptr;
    A.natom = c->natom;
    A.mol_atoms = c->nmol > 1 ? c->d_mol_atoms.p : nullptr;
    A.boys = c->d_boys.p;
    A.nbf = c->nbf;
    return A;
}

// One-electron integrals of the basis on the shell-pair kernels: S, T, V
// (N x N) and, when M and Lm are given, the dipole and angular-momentum
// integrals about `center`.  A basis of several molecules gets only the
// molecules' own blocks; the rest of the outputs is cleared.
int one_electron_shells(mmd_ctx* c, const double center[3], double* S, double* T, double* V, double* M, double* Lm)
{
    if (int rc = onee_pair_list(c)) return rc;
    const size_t nn = (size_t)c->nbf * c->nbf;
    if (c->nmol > 1) {
        for (double* x : {S, T, V}) HIP_TRY(launch_fill(nn, x, 0.0, c->st));
        if (M && Lm)
            for (double* x : {M, Lm}) HIP_TRY(launch_fill(3 * nn, x, 0.0, c->st));
    }
    OneeArgs A = onee_args(c);
    A.cx = center[0];
    A.cy = center[1];
    A.cz = center[2];
    A.S = S;
    A.T = T;
    A.V = V;
    A.M = M;
    A.Lm = Lm;
    HIP_TRY(launch_one_electron_shells(A, c->d_onee_list.p, c->onee_off, c->st));
    return MMD_OK;
}

// The Schwarz diagonal (pq|pq) of the basis into out (N x N; for several
// molecules, zero outside their blocks): shell-pair kernels where the basis
// forms complete shells, else the per-function kernel.
int schwarz_diagonal(mmd_ctx* c, double* out)
{
    const int N = c->nbf;
    if (!c->shells_ok) {
        HIP_TRY(launch_eri_diag(N, c->d_bf.p, c->d_bf_exp.p, c->d_bf_w.p, c->d_boys.p, out, c->st,
                                c->nmol > 1 ? c->d_plist.p : nullptr, c->npl));
        return MMD_OK;
    }
    if (int rc = onee_pair_list(c)) return rc;
    if (c->nmol > 1) HIP_TRY(launch_fill((size_t)N * N, out, 0.0, c->st));
    HIP_TRY(launch_schwarz_shells(onee_args(c), c->d_onee_list.p, c->onee_off, out, c->st));
    return MMD_OK;
}

void class_of(int qc, int* pcb, int* pck);

// Shell pairs of each molecule, grouped by pair class and sorted in each
// class by (molecule, primitive pairs descending, Schwarz factor
// descending), with their primitive-pair tables, on the device.  diag: the
// N x N Schwarz diagonal (pq|pq) on the device, or null before it is known
// (factors 1).  With a diagonal also the Fock build's work units: they belong
// to the pair table, and a build (mmd_fock_delta_noalloc) allocates nothing.
int build_pairs(mmd_ctx* c, const double* diag)
{
    if (int rc = onee_pair_list(c)) return rc;
    c->grad_plan_ok = false;
    c->btab_ok = c->qraw_ok = false;
    c->pairs_ok = c->units_ok = false;
    for (int pc = 0; pc <= NPAIRCLASS; ++pc) c->pc_off[pc] = c->onee_off[pc];
    const size_t n = (size_t)c->pc_off[NPAIRCLASS];
    HIP_TRY(c->d_pairs.reserve(n));
    HIP_TRY(c->w_count.reserve(n));
    HIP_TRY(c->w_entry.reserve(n));
    HIP_TRY(c->w_q.reserve(n));
    HIP_TRY(c->w_scan.reserve(n + n / 1024 + 2));
    int maxnp = 1;
    for (const Shell& s : c->shells) maxnp = std::max(maxnp, s.np);
    HIP_TRY(c->w_keep.reserve(n * pair_keep_pieces(maxnp)));
    constexpr int HEAD = (PAIR_REPORT + UNIT_HIST + 1) & ~1;   // the bound after it is 8 bytes
    HIP_TRY(c->w_ints.reserve(HEAD + 2));
    PairInput I;
    I.shells = c->d_oshell.p;
    I.exps = c->d_sh_exp.p;
    I.wts = c->d_sh_w.p;
    I.list = c->d_onee_list.p;
    I.ranges = c->d_ranges.p;
    I.mol_blocks = c->nmol > 1 ? c->d_mol_blocks.p : nullptr;
    I.diag = diag;
    I.nmol = c->nmol;
    I.N = c->nbf;
    PairWork W;
    W.count = c->w_count.p;
    W.entry = c->w_entry.p;
    W.q = c->w_q.p;
    W.scan = c->w_scan.p;
    W.keep = c->w_keep.p;
    W.report = c->w_ints.p;
    W.hist = W.report + PAIR_REPORT;
    W.qmax = reinterpret_cast<unsigned long long*>(W.report + HEAD);
    W.nclear = HEAD + 2;
    UnitInput U;
    U.pairs = c->d_pairs.p;
    U.ranges = c->d_ranges.p;
    U.nmol = c->nmol;
    for (int pc = 0; pc <= NPAIRCLASS; ++pc) I.off[pc] = U.off[pc] = c->pc_off[pc];
    // quartet-class sizes (implicit enumeration; for several molecules an
    // upper bound, the screen keeps the quartets of one molecule)
    c->qc_off[0] = 0;
    for (int qc = 0; qc < NQCLASS; ++qc) {
        int pcb, pck;
        class_of(qc, &pcb, &pck);
        const int64_t nb = c->pc_off[pcb + 1] - c->pc_off[pcb];
        const int64_t nk = c->pc_off[pck + 1] - c->pc_off[pck];
        c->qc_total[qc] = (pcb == pck) ? nb * (nb + 1) / 2 : nb * nk;
        c->qc_off[qc + 1] = c->qc_off[qc] + c->qc_total[qc];
        // ket segment of a work unit: long (survivors are batched inside a
        // unit), but short enough for a few thousand segments per class.
        // (Shorter segments make a class that runs alone faster, but cost
        // more than they gain when classes or molecules share the GPU.)
        int seg = 4096;
        while (seg > 256 && c->qc_total[qc] / std::max(1, c->nmol) / seg < 4096) seg /= 2;
        // One small molecule leaves most of the GPU idle, and a class lasts as
        // long as its longest unit: segments of down to 32 kets until the
        // class has about 512.  (H2O)2, 3 and 5 in 6-31G, 6-31G* and 6-31G
        // 158, 423 and 239 us per build without, 137, 356 and 204 with; more
        // units cost more than they gain ((H2O)5 204, 234, 256, 296 us for
        // 512, 1024, 2048, 4096; (H2O)8 cc-pVDZ 1.76, 1.88, 2.07, 2.37 ms).
        if (c->nmol == 1)
            while (seg > 32 && c->qc_total[qc] / seg < 512) seg /= 2;
        U.seg[qc] = seg;
    }
    HIP_TRY(launch_pair_sort(I, W, U, diag != nullptr, c->d_pairs.p, c->st));
    // Sizes of the tables: as if no primitive pair were screened out, so that
    // the device need not be waited for between the sort and the tables; the
    // counts themselves where that could waste more than TABLE_SLACK bytes.
    size_t npp = 0, units = 0;
    for (int pc = 0; pc < NPAIRCLASS; ++pc) npp += (size_t)c->pair_prims[pc];
    if (diag)
        for (int qc = 0; qc < NQCLASS; ++qc) {
            int pcb, pck;
            class_of(qc, &pcb, &pck);
            for (int m = 0; m < c->nmol; ++m) {
                const int2 r = c->pair_ranges[(size_t)pck * c->nmol + m];
                units += (size_t)c->pair_slices[(size_t)pcb * c->nmol + m]
                       * (size_t)((r.y - r.x + U.seg[qc] - 1) / U.seg[qc]);
            }
        }
    constexpr size_t TABLE_SLACK = (size_t)64 << 20;
    if (npp * (sizeof(PrimPair) + sizeof(double) * (1 + KET_FIELDS)) + units * (sizeof(int4) + sizeof(UnitBound))
        > TABLE_SLACK) {
        int h[PAIR_REPORT];
        HIP_TRY(hipMemcpyAsync(h, W.report, sizeof(h), hipMemcpyDeviceToHost, c->st));
        HIP_TRY(hipStreamSynchronize(c->st));
        PairStats stats;
        memcpy(&stats, h, sizeof(stats));
        npp = units = 0;
        for (int pc = 0; pc < NPAIRCLASS; ++pc) npp += (size_t)stats.total[pc];
        if (diag)
            for (int qc = 0; qc < NQCLASS; ++qc) units += (size_t)h[PAIR_STATS + qc];
    }
    npp = std::max<size_t>(1, npp);
    units = std::max<size_t>(1, units);
    HIP_TRY(c->d_pp.reserve(npp));
    HIP_TRY(c->d_ppa.reserve(npp));
    c->kpp_stride = (int64_t)((npp + 15) & ~(size_t)15);   // fields start on cache lines
    HIP_TRY(c->d_kscr.reserve(n));
    HIP_TRY(c->d_kref.reserve(n));
    HIP_TRY(c->d_kpp.reserve((size_t)(KET_FIELDS * c->kpp_stride)));
    const KetTables K = {c->d_kscr.p, c->d_kref.p, c->d_kpp.p, c->kpp_stride};
    UnitTables T = {nullptr, nullptr};
    if (diag) {
        HIP_TRY(c->d_units.reserve(units));
        HIP_TRY(c->d_ubound.reserve(units));
        if (c->nmol > 1) HIP_TRY(c->d_live.reserve(units));
        T = {c->d_units.p, c->d_ubound.p};
    }
    HIP_TRY(launch_pair_tables(I, W, c->d_pairs.p, c->d_pp.p, c->d_ppa.p, K, U, T, c->h_pairs, c->st));
    HIP_TRY(hipStreamSynchronize(c->st));
    PairStats stats;
    memcpy(&stats, c->h_pairs, sizeof(stats));
    for (int pc = 0; pc < NPAIRCLASS; ++pc) {
        c->pc_npp[pc] = stats.total[pc];
        c->pc_maxpp[pc] = std::max(1, stats.maxpp[pc]);
    }
    if (diag) {
        c->unit_off[0] = 0;
        for (int qc = 0; qc < NQCLASS; ++qc) c->unit_off[qc + 1] = c->unit_off[qc] + c->h_pairs[PAIR_STATS + qc];
        c->units_ok = true;
    }
    HIP_TRY(c->d_ctr.reserve(1));
    c->pairs_ok = true;
    for (int qc = 0; qc < NQCLASS; ++qc) {
        c->plan_ms[qc] = 0.0;
        c->impl_choice[qc] = -1;
    }
    c->plan_countdown = 0;
    c->tune_phase = 0;
    return MMD_OK;
}

void class_of(int qc, int* pcb, int* pck)
{
    int b = 0;
    while ((b + 1) * (b + 2) / 2 <= qc) ++b;
    *pcb = b;
    *pck = qc - b * (b + 1) / 2;
}

int grid_for(int64_t items)
{
    int64_t g = (items + 255) / 256;
    if (g < 1) g = 1;
    if (g > 2048) g = 2048;
    return (int)g;
}

// The side streams of n streams, created when a basis is set: HIP
// deals streams to its few hardware queues in order of creation, so contexts
// that each made all seven at once had their main streams on one queue, and
// batch groups on different contexts ran one after the other.
int ensure_streams(mmd_ctx* c, int n)
{
    for (int i = 0; i + 1 < n; ++i) {
        if (!c->side[i]) HIP_TRY(hipStreamCreateWithFlags(&c->side[i], hipStreamNonBlocking));
        if (!c->evjoin[i]) HIP_TRY(hipEventCreateWithFlags(&c->evjoin[i], hipEventDisableTiming));
    }
    return MMD_OK;
}

// Independent launches spread over the context's streams, largest first and
// each to the least loaded stream, between a fork from and a join to c->st.
struct StreamTask {
    double cost;
    int id;
};
template <class F>
int spread_tasks(mmd_ctx* c, std::vector<StreamTask>& tasks, F&& launch)
{
    std::sort(tasks.begin(), tasks.end(), [](const StreamTask& x, const StreamTask& y) { return x.cost > y.cost; });
    hipStream_t streams[1 + mmd_ctx::NSIDE] = {c->st};
    for (int i = 0; i < mmd_ctx::NSIDE; ++i) streams[1 + i] = c->side[i];
    double load[1 + mmd_ctx::NSIDE] = {0};
    bool used[1 + mmd_ctx::NSIDE] = {true};
    HIP_TRY(hipEventRecord(c->evfork, c->st));
    for (const StreamTask& t : tasks) {
        int si = 0;
        for (int i = 1; i < c->nstreams; ++i)
            if (load[i] < load[si]) si = i;
        load[si] += t.cost;
        if (!used[si]) {
            HIP_TRY(hipStreamWaitEvent(streams[si], c->evfork, 0));
            used[si] = true;
        }
        HIP_TRY(launch(t.id, streams[si]));
    }
    for (int i = 1; i < c->nstreams; ++i) {
        if (!used[i]) continue;
        HIP_TRY(hipEventRecord(c->evjoin[i - 1], streams[i]));
        HIP_TRY(hipStreamWaitEvent(c->st, c->evjoin[i - 1], 0));
    }
    return MMD_OK;
}

ClassArgs base_args(mmd_ctx* c)
{
    ClassArgs A;
    memset(&A, 0, sizeof(A));
    A.pairs = c->d_pairs.p;
    A.pp = c->d_pp.p;
    A.boys = c->d_boys.p;
    A.boysf = c->d_boysf.p;
    A.gcomp = c->d_gcomp.p;
    A.N = c->nbf;
    return A;
}

// Device memory a Fock build works in besides its inputs and outputs: work-unit
// counters, survivor counts and statistics, the shell-block maxima of |dP|,
// and the survivor lists of the classes that run on the wavefront-per-quartet
// kernel (class qc at surv + surv_off[qc]).  The context's buffers, or a
// caller-free static array (mmd_fock_delta_noalloc).
struct FockScratch {
    int (*rowctr)[ROW_QUEUES * ROW_QUEUE_PAD] = nullptr;   // cleared, with the others, by the build's preparation kernel
    int* count = nullptr;
    const int* nlive = nullptr;
    // NPRIM_SLOTS counters: primitive quartets (FP64 tier), shell quartets of
    // the row kernels (FP64, FP32 tier), primitive quartets (FP32 tier)
    unsigned long long* nprim = nullptr;
    void counters(FockCounters* c)
    {
        rowctr = c->rowctr;
        count = c->count;
        nprim = c->nprim;
        nlive = c->nlive;
    }
    double* Dsh = nullptr;                 // nshell^2
    const int* live = nullptr;             // batches: the build's live units (launch_unit_live)
    int2* surv = nullptr;
    int64_t surv_off[NQCLASS] = {0};       // survivor lists, packed: wave classes only
    int64_t surv_cap = -1;                 // entries available at surv; < 0: grow the context's buffer
    bool allow_measure = true;             // may create events and re-measure the stream plan
    bool profile_events = false;           // with profiling on, time the classes even without allow_measure
};

// Launch the Fock kernels of every class.  Classes with a row kernel screen
// inline; the wavefront-per-quartet classes (and any class whose bra rows do
// not fit in LDS) are screened into survivor lists first.
int run_fock_classes(mmd_ctx* c, ClassArgs A, double tol, FockScratch& W0)
{
    const bool tier32 = c->fp32_below > tol;
    if (!c->units_ok) return fail(MMD_ERR_STATE, "work units are built by mmd_schwarz / mmd_set_schwarz");
    bool row_kernel[NQCLASS], kj_lds[NQCLASS];
    int maxpp[NQCLASS];
    // a build that times the row or the matrix-core variant of the classes
    // that have both, while some of them are undecided
    bool tuning = false;
    if (c->impl_mode == 2 && W0.allow_measure)
        for (int qc = 0; qc < NQCLASS; ++qc) {
            int la, lb, lc, ld;
            qclass_decode(qc, &la, &lb, &lc, &ld);
            if (c->qc_total[qc] && fock_class_has_both(la, lb, lc, ld) && c->impl_choice[qc] < 0) tuning = true;
        }
    for (int qc = 0; qc < NQCLASS; ++qc) {
        int la, lb, lc, ld, pcb, pck;
        qclass_decode(qc, &la, &lb, &lc, &ld);
        class_of(qc, &pcb, &pck);
        maxpp[qc] = c->pc_maxpp[pcb];
        bool mfma = fock_class_is_wave(la, lb, lc, ld);
        if (mfma && fock_class_has_both(la, lb, lc, ld)) {
            if (c->impl_mode == 0) mfma = false;
            else if (c->impl_mode == 2 && c->impl_choice[qc] >= 0) mfma = c->impl_choice[qc] == 1;
            else if (c->impl_mode == 2 && tuning) mfma = c->tune_phase == 1;
        }
        // the ket-side Coulomb buffer where it fits in 64 KiB (two workgroups
        // per CU and more); the row kernel without it up to the device's LDS
        // ((dd|ss) at 400 functions, 78 KiB: 0.25 ms against 12.6 on the
        // generic kernel); else the wavefront-per-quartet kernel
        kj_lds[qc] = fock_class_lds(qc, 0, c->rw, maxpp[qc], 1) <= std::min<size_t>(c->max_lds, 65536);
        row_kernel[qc] = !mfma && (kj_lds[qc] || fock_class_lds(qc, 0, c->rw, maxpp[qc], 0) <= c->max_lds);
    }
    c->tune_measuring = tuning;
    {
        // survivor lists only for the classes that use them, packed; with the
        // FP32 tier each class has a second list right after the first
        int64_t off = 0;
        for (int qc = 0; qc < NQCLASS; ++qc) {
            W0.surv_off[qc] = off;
            if (c->qc_total[qc] && !row_kernel[qc]) off += (tier32 ? 2 : 1) * c->qc_total[qc];
        }
        if (W0.surv_cap < 0) {
            HIP_TRY(c->d_surv.reserve((size_t)std::max<int64_t>(off, 1)));
            W0.surv = c->d_surv.p;
        } else if (off > W0.surv_cap) {
            return fail(MMD_ERR_ARG, "survivor lists need %lld entries, the scratch holds %lld", (long long)off,
                        (long long)W0.surv_cap);
        }
    }
    // Classes run concurrently on the main and side streams (longest first,
    // each to the least loaded stream), so that the small classes fill the
    // GPU beside the large ones.  Profiling mode 1 brackets every class with
    // events on its own stream (times include sharing the GPU with the other
    // classes); mode 2 runs the classes one after the other on the main
    // stream, so that each class's events time it alone.
    int order[NQCLASS], nord = 0;
    double cost[NQCLASS] = {0};
    for (int qc = 0; qc < NQCLASS; ++qc) {
        if (c->qc_total[qc] == 0) continue;
        int pcb, pck, la, lb, lc, ld;
        class_of(qc, &pcb, &pck);
        qclass_decode(qc, &la, &lb, &lc, &ld);
        const double prim = (double)c->pc_npp[pcb] * c->pc_npp[pck] * (pcb == pck ? 0.5 : 1.0);
        const int L = la + lb + lc + ld;
        cost[qc] = prim * (40.0 + 4.0 * nherm(L) + (double)ncart(la) * ncart(lb) * ncart(lc) * ncart(ld));
        order[nord++] = qc;
    }
    const int nstream = c->profiling == 2 ? 1 : c->nstreams;
    // Plan on the measured class durations once they exist: the model above
    // misses the latency floor of the small classes (150-300 us each at
    // (H2O)8/cc-pVDZ, whatever their work), which left the longest stream
    // twice as long as the others.  One build in PLAN_EVERY measures again.
    const bool measure = (W0.allow_measure && c->profiling == 0 && nstream > 1 && c->plan_countdown <= 0) || tuning;
    bool measured = nord > 0;
    for (int oi = 0; oi < nord; ++oi) measured = measured && c->plan_ms[order[oi]] > 0.0;
    if (measured)
        for (int oi = 0; oi < nord; ++oi) cost[order[oi]] = c->plan_ms[order[oi]];
    if ((measure || (c->profiling && W0.profile_events)) && !c->evc[0])
        for (int i = 0; i < 3 * NQCLASS; ++i) HIP_TRY(hipEventCreate(&c->evc[i]));
    c->plan_measuring = measure;
    std::sort(order, order + nord, [&](int x, int y) { return cost[x] > cost[y]; });
    hipStream_t streams[1 + mmd_ctx::NSIDE] = {c->st};
    for (int i = 0; i < mmd_ctx::NSIDE; ++i) streams[1 + i] = c->side[i];
    double load[1 + mmd_ctx::NSIDE] = {0};
    bool used[1 + mmd_ctx::NSIDE] = {true};
    if (nstream > 1) HIP_TRY(hipEventRecord(c->evfork, c->st));
    for (int oi = 0; oi < nord; ++oi) {
        const int qc = order[oi];
        int si = 0;
        for (int i = 1; i < nstream; ++i)
            if (load[i] < load[si]) si = i;
        load[si] += cost[qc];
        hipStream_t sq = streams[si];
        if (!used[si]) {
            HIP_TRY(hipStreamWaitEvent(sq, c->evfork, 0));
            used[si] = true;
        }
        int pcb, pck, la, lb, lc, ld;
        class_of(qc, &pcb, &pck);
        qclass_decode(qc, &la, &lb, &lc, &ld);
        const int nb = c->pc_off[pcb + 1] - c->pc_off[pcb];
        const int nk = c->pc_off[pck + 1] - c->pc_off[pck];
        const bool events = measure || (c->profiling && (W0.allow_measure || W0.profile_events));
        if (events) HIP_TRY(hipEventRecord(c->evc[3 * qc], sq));
        if (row_kernel[qc]) {
            RowArgs R;
            R.boff = c->pc_off[pcb];
            R.nb = nb;
            R.koff = c->pc_off[pck];
            R.nk = nk;
            R.tri = pcb == pck ? 1 : 0;
            R.nshell = (int)c->shells.size();
            R.Dsh = W0.Dsh;
            R.live = W0.live ? W0.live + c->unit_off[qc] : nullptr;
            R.nlive = W0.nlive + qc;
            R.row_counter = W0.rowctr[qc];
            R.maxpp = maxpp[qc];
            R.kj = kj_lds[qc] ? 1 : 0;
            R.kslice = c->ket_slice[qc];
            R.rw = c->rw;
            R.kscr = c->d_kscr.p;
            R.kref = c->d_kref.p;
            R.kpp = c->d_kpp.p;
            R.kstride = c->kpp_stride;
            R.units = c->d_units.p + c->unit_off[qc];
            const int64_t units = c->unit_off[qc + 1] - c->unit_off[qc];
            R.nunits = (int)units;
            if (units == 0) {
                if (events) {
                    HIP_TRY(hipEventRecord(c->evc[3 * qc + 1], sq));
                    HIP_TRY(hipEventRecord(c->evc[3 * qc + 2], sq));
                }
                continue;
            }
            R.stat_nquart = W0.nprim + NQCLASS + qc;
            R.stat_nprim = c->profiling ? W0.nprim + qc : nullptr;
            R.tier_lo = tier32 ? c->fp32_below : 0.0;
            R.tier_hi = HUGE_VAL;
            const int grid = (int)std::min<int64_t>(units, 2048);
            HIP_TRY(launch_fock_class(qc, 0, A, R, grid, sq));
            if (events) HIP_TRY(hipEventRecord(c->evc[3 * qc + 1], sq));
            if (tier32) {
                // FP32 tier: the same units, quartets with tol <= bound < fp32_below
                R.tier_lo = 0.0;
                R.tier_hi = c->fp32_below;
                R.row_counter = W0.rowctr[NQCLASS + qc];
                R.stat_nquart = W0.nprim + 2 * NQCLASS + qc;
                R.stat_nprim = c->profiling ? W0.nprim + 3 * NQCLASS + qc : nullptr;
                // the second traversal holds the many small-bound quartets
                // of a unit: longer ket slices keep its items few ((H2O)16
                // cc-pVDZ tier build 9.3 ms with the FP64 pass's slices of 2,
                // 8.8 ms with 8)
                R.kslice = std::max(R.kslice, 8);
                HIP_TRY(launch_fock_class(qc, 1, A, R, grid, sq));
            }
        } else {
            // one screening pass; with the FP32 tier the quartets with bound
            // in [tol, fp32_below) go to a second list and run in FP32
            int2* surv = W0.surv + W0.surv_off[qc];
            int2* surv32 = tier32 ? surv + c->qc_total[qc] : nullptr;
            HIP_TRY(launch_screen_class(c->pc_off[pcb], nb, c->pc_off[pck], nk, pcb == pck ? 1 : 0, c->d_pairs.p,
                                        W0.Dsh, (int)c->shells.size(), tol, 0, surv, W0.count + qc, sq,
                                        c->fp32_below, surv32, W0.count + NQCLASS + qc));
            ClassArgs W = A;
            W.quart = surv;
            W.count = W0.count + qc;
            if (c->profiling)
                HIP_TRY(launch_count_prims(W.quart, W.count, c->d_pairs.p, W0.nprim + qc, sq));
            HIP_TRY(launch_fock_wave_class(la, lb, lc, ld, 0, W, c->qc_total[qc], sq));
            if (events) HIP_TRY(hipEventRecord(c->evc[3 * qc + 1], sq));
            if (tier32) {
                W.quart = surv32;
                W.count = W0.count + NQCLASS + qc;
                if (c->profiling)
                    HIP_TRY(launch_count_prims(W.quart, W.count, c->d_pairs.p, W0.nprim + 3 * NQCLASS + qc, sq));
                HIP_TRY(launch_fock_wave_class(la, lb, lc, ld, 1, W, c->qc_total[qc], sq));
            }
        }
        if (events) HIP_TRY(hipEventRecord(c->evc[3 * qc + 2], sq));
    }
    for (int i = 1; i < nstream; ++i) {
        if (!used[i]) continue;
        HIP_TRY(hipEventRecord(c->evjoin[i - 1], streams[i]));
        HIP_TRY(hipStreamWaitEvent(c->st, c->evjoin[i - 1], 0));
    }
    for (int qc = 0; qc < NQCLASS; ++qc) c->last_row_kernel[qc] = row_kernel[qc];
    return MMD_OK;
}

// Survivors of the build whose counters are in h_ctr: per-class lists (wave
// classes) and FP64 and FP32 row-kernel counts.
void count_survivors(mmd_ctx* c)
{
    const int* h = c->h_ctr->count;
    const unsigned long long* hq = c->h_ctr->nprim + NQCLASS;
    int64_t s = 0, s32 = 0;
    for (int i = 0; i < NQCLASS; ++i) {
        s += (int64_t)h[i] + (int64_t)h[NQCLASS + i] + (int64_t)hq[i] + (int64_t)hq[NQCLASS + i];
        s32 += (int64_t)h[NQCLASS + i] + (int64_t)hq[NQCLASS + i];
    }
    c->last_nsurv = s;
    c->last_nsurv_fp32 = s32;
}

// Per-class statistics and event times of the last build (profiling on),
// also added to the sums since profiling was turned on.  Called after the
// build's end event, so the readback is not timed.
int collect_profile(mmd_ctx* c)
{
    HIP_TRY(hipMemcpyAsync(c->h_ctr, c->d_ctr.p, sizeof(FockCounters), hipMemcpyDeviceToHost, c->st));
    HIP_TRY(hipStreamSynchronize(c->st));
    const int* h = c->h_ctr->count;
    const unsigned long long* hp = c->h_ctr->nprim;
    for (int qc = 0; qc < NQCLASS; ++qc) {
        if (!c->qc_total[qc]) {
            c->st_nquart[qc] = c->st_nprim[qc] = 0;
            c->st_ms[qc] = 0.0;
            continue;
        }
        const int64_t q64 = c->last_row_kernel[qc] ? (int64_t)hp[NQCLASS + qc] : (int64_t)h[qc];
        const int64_t q32 = c->last_row_kernel[qc] ? (int64_t)hp[2 * NQCLASS + qc] : (int64_t)h[NQCLASS + qc];
        c->st_nquart[qc] = q64 + q32;
        c->st_nprim[qc] = (int64_t)(hp[qc] + hp[3 * NQCLASS + qc]);
        float ms = 0.f, ms64 = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, c->evc[3 * qc], c->evc[3 * qc + 2]));
        HIP_TRY(hipEventElapsedTime(&ms64, c->evc[3 * qc], c->evc[3 * qc + 1]));
        c->st_ms[qc] = ms;
        ProfileSum& a = c->psum[qc];
        a.nquart[0] += q64;
        a.nquart[1] += q32;
        a.nprim[0] += (int64_t)hp[qc];
        a.nprim[1] += (int64_t)hp[3 * NQCLASS + qc];
        a.ms[0] += ms64;
        a.ms[1] += ms - ms64;
        a.builds += 1;
    }
    return MMD_OK;
}

}  // namespace

namespace {
// The Schwarz matrix (pq|pq) is in d_schwarz: its square roots for the
// screen, and the sorted shell-pair tables with their factors
// q = max sqrt((ab|ab)) and the work units.
int finish_schwarz(mmd_ctx* ctx)
{
    const size_t nn = (size_t)ctx->nbf * ctx->nbf;
    HIP_TRY(launch_sqrt_clamped(nn, ctx->d_schwarz.p, ctx->d_sqS.p, ctx->st));
    if (ctx->shells_ok) {   // else only the per-function paths are available
        if (int rc = build_pairs(ctx, ctx->d_schwarz.p)) return rc;
    } else {
        HIP_TRY(hipStreamSynchronize(ctx->st));
    }
    ctx->schwarz_ok = true;
    return MMD_OK;
}

}  // namespace

namespace mmd {
void set_last_error(const char* msg) { g_last_error = msg; }
}  // namespace mmd

// ===========================================================================
// C ABI
// ===========================================================================
extern "C" {

const char* mmd_last_error(void) { return g_last_error.c_str(); }

int mmd_version(void) { return 1; }

int mmd_device_count(int* count)
{
    if (!count) return fail(MMD_ERR_ARG, "null pointer");
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess) n = 0;
    *count = n;
    return MMD_OK;
}

int mmd_ctx_create(mmd_ctx** out, int device_id)
{
    if (!out) return fail(MMD_ERR_ARG, "null output pointer");
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return fail(MMD_ERR_DEVICE, "no HIP device available");
    if (device_id < 0 || device_id >= n) return fail(MMD_ERR_ARG, "device %d out of range (%d devices)", device_id, n);
    HIP_TRY(hipSetDevice(device_id));
    mmd_ctx* c = new (std::nothrow) mmd_ctx();
    if (!c) return fail(MMD_ERR_NOMEM, "context allocation failed");
    c->device = device_id;
    for (int qc = 0; qc < NQCLASS; ++qc) {
        c->impl_choice[qc] = -1;
        c->ket_slice[qc] = KSLICE_DEFAULT;
    }
    // Classes on more streams than the process has hardware queues would
    // share queues in an order the longest-first plan does not see: spread
    // them over min(8, GPU_MAX_HW_QUEUES) streams (HIP's default is 4).  The
    // variable is read once, at the first context of the process, so that a
    // later change of the environment (after HIP read it) does not matter.
    {
        static const int hw_queues = [] {
            const char* hq = getenv("GPU_MAX_HW_QUEUES");
            const int q = hq ? atoi(hq) : 4;
            return q > 0 ? q : 4;
        }();
        c->nstreams = std::max(1, std::min(hw_queues, 1 + mmd_ctx::NSIDE));
    }
    int lds_max = 0;
    if (hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, device_id) == hipSuccess &&
        lds_max > 0)
        c->max_lds = (size_t)lds_max;
    c->max_lds_device = c->max_lds;
    if (lds_max > 0) c->lds_per_block = (size_t)lds_max;
    hipError_t e = hipStreamCreateWithFlags(&c->st, hipStreamNonBlocking);
    if (e == hipSuccess) {
        std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
        e = hipHostMalloc((void**)&c->h_ctr, sizeof(FockCounters) + sizeof(int) * PAIR_REPORT, hipHostMallocDefault);
        if (e == hipSuccess) c->h_pairs = reinterpret_cast<int*>(c->h_ctr + 1);
    }
    if (e == hipSuccess) e = hipEventCreate(&c->ev0);
    if (e == hipSuccess) e = hipEventCreate(&c->ev1);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&c->evfork, hipEventDisableTiming);
    std::vector<double> tab;
    boys_build_table(tab);
    if (e == hipSuccess) e = c->d_boys.reserve(tab.size());
    if (e == hipSuccess)
        e = hipMemcpyAsync(c->d_boys.p, tab.data(), sizeof(double) * tab.size(), hipMemcpyHostToDevice, c->st);
    std::vector<float> tabf(tab.begin(), tab.end());
    if (e == hipSuccess) e = c->d_boysf.reserve(tabf.size());
    if (e == hipSuccess)
        e = hipMemcpyAsync(c->d_boysf.p, tabf.data(), sizeof(float) * tabf.size(), hipMemcpyHostToDevice, c->st);
    if (e == hipSuccess) e = hipStreamSynchronize(c->st);
    if (e != hipSuccess) {
        mmd_ctx_destroy(c);
        return fail(MMD_ERR_DEVICE, "context setup: %s", hipGetErrorString(e));
    }
    // this device's address of the static scratch (once per device)
    const int rc = scratch_for_device(device_id, &c->noalloc_scratch);
    if (rc) {
        mmd_ctx_destroy(c);
        return rc;
    }
    *out = c;
    return MMD_OK;
}

int mmd_release_workspaces(int device_id)
{
    int n = 0;
    (void)mmd_device_count(&n);
    if (device_id < 0 || device_id >= n) return fail(MMD_ERR_ARG, "device id out of range");
    HIP_TRY(hipSetDevice(device_id));
    (void)pool_release(device_id);
    return MMD_OK;
}

void mmd_ctx_destroy(mmd_ctx* ctx)
{
    if (!ctx) return;
    (void)hipSetDevice(ctx->device);
    if (ctx->st) (void)hipStreamSynchronize(ctx->st);
    if (ctx->ev0) (void)hipEventDestroy(ctx->ev0);
    if (ctx->ev1) (void)hipEventDestroy(ctx->ev1);
    for (int i = 0; i < 3 * NQCLASS; ++i)
        if (ctx->evc[i]) (void)hipEventDestroy(ctx->evc[i]);
    for (int i = 0; i < mmd_ctx::NSIDE; ++i) {
        if (ctx->side[i]) (void)hipStreamSynchronize(ctx->side[i]);
        if (ctx->evjoin[i]) (void)hipEventDestroy(ctx->evjoin[i]);
        if (ctx->side[i]) (void)hipStreamDestroy(ctx->side[i]);
    }
    if (ctx->evfork) (void)hipEventDestroy(ctx->evfork);
    std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
    if (ctx->blas) (void)rocblas_destroy_handle(ctx->blas);
    if (ctx->h_ctr) (void)hipHostFree(ctx->h_ctr);
    hipStream_t st = ctx->st;
    delete ctx;  // frees device buffers
    if (st) (void)hipStreamDestroy(st);
}

int mmd_set_basis(mmd_ctx* ctx, int nbf, const double* origin, const int32_t* lmn, const int32_t* nprim,
                  const double* exps, const double* weights)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (nbf <= 0 || !origin || !lmn || !nprim || !exps || !weights) return fail(MMD_ERR_ARG, "invalid basis arguments");
    if ((rc = ensure_streams(ctx, ctx->nstreams))) return rc;   // a context with a basis has its streams
    ctx->bf.assign(nbf, BFDesc{});
    ctx->bf_exp.clear();
    ctx->bf_w.clear();
    for (int i = 0; i < nbf; ++i) {
        BFDesc& b = ctx->bf[i];
        b.x = origin[3 * i];
        b.y = origin[3 * i + 1];
        b.z = origin[3 * i + 2];
        b.l = lmn[3 * i];
        b.m = lmn[3 * i + 1];
        b.n = lmn[3 * i + 2];
        if (b.l < 0 || b.m < 0 || b.n < 0) return fail(MMD_ERR_ARG, "negative angular exponent");
        if (b.l + b.m + b.n > MAX_L)
            return fail(MMD_ERR_UNSUPPORTED, "basis function %d has l=%d; this build supports l <= %d", i,
                        b.l + b.m + b.n, MAX_L);
        if (nprim[i] <= 0) return fail(MMD_ERR_ARG, "basis function %d has no primitives", i);
        b.np = nprim[i];
        b.p0 = (int)ctx->bf_exp.size();
        b.pad = 0;
        for (int p = 0; p < b.np; ++p) {
            const double e = exps[b.p0 + p];
            if (!(e > 0.0)) return fail(MMD_ERR_ARG, "non-positive exponent");
            ctx->bf_exp.push_back(e);
            ctx->bf_w.push_back(weights[b.p0 + p]);
        }
    }
    ctx->nbf = nbf;
    ctx->pairs_ok = false;
    ctx->schwarz_ok = false;
    ctx->nmol = 1;
    ctx->mol_f0.assign(1, 0);
    ctx->mol_n.assign(1, nbf);
    ctx->mol_atoms.clear();
    ctx->npl = 0;
    ctx->rw = nbf;
    HIP_TRY(ctx->d_bf.reserve(nbf));
    HIP_TRY(ctx->d_bf_exp.reserve(ctx->bf_exp.size()));
    HIP_TRY(ctx->d_bf_w.reserve(ctx->bf_w.size()));
    HIP_TRY(hipMemcpyAsync(ctx->d_bf.p, ctx->bf.data(), sizeof(BFDesc) * nbf, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(ctx->d_bf_exp.p, ctx->bf_exp.data(), sizeof(double) * ctx->bf_exp.size(),
                           hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(ctx->d_bf_w.p, ctx->bf_w.data(), sizeof(double) * ctx->bf_w.size(), hipMemcpyHostToDevice,
                           ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    build_shells(ctx);
    if (ctx->shells_ok) {
        rc = upload_shells(ctx);
        if (rc) return rc;
    }
    const size_t nn = (size_t)nbf * nbf;
    HIP_TRY(ctx->d_D.reserve(nn));
    HIP_TRY(ctx->d_Dim.reserve(nn));
    HIP_TRY(ctx->d_absD.reserve(nn));
    HIP_TRY(ctx->d_G.reserve(nn));
    HIP_TRY(ctx->d_Gout.reserve(nn));
    HIP_TRY(ctx->d_schwarz.reserve(nn));
    HIP_TRY(ctx->d_sqS.reserve(nn));
    const size_t ns = ctx->shells.size();
    HIP_TRY(ctx->d_Dsh.reserve(ns * ns));
    return MMD_OK;
}

int mmd_set_atoms(mmd_ctx* ctx, int natom, const double* Z, const double* xyz)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (natom < 0 || (natom > 0 && (!Z || !xyz))) return fail(MMD_ERR_ARG, "invalid atoms");
    std::vector<double> a(4 * (size_t)std::max(natom, 1));
    for (int i = 0; i < natom; ++i) {
        a[4 * i] = Z[i];
        a[4 * i + 1] = xyz[3 * i];
        a[4 * i + 2] = xyz[3 * i + 1];
        a[4 * i + 3] = xyz[3 * i + 2];
    }
    HIP_TRY(ctx->d_atoms.reserve(a.size()));
    HIP_TRY(hipMemcpyAsync(ctx->d_atoms.p, a.data(), sizeof(double) * a.size(), hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    ctx->natom = natom;
    return MMD_OK;
}

int mmd_set_molecules(mmd_ctx* ctx, int nmol, const int32_t* nbf_per_mol, const int32_t* natom_per_mol)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (ctx->nbf == 0) return fail(MMD_ERR_STATE, "no basis set");
    if (nmol < 1 || !nbf_per_mol || !natom_per_mol) return fail(MMD_ERR_ARG, "invalid molecule arguments");
    int64_t sf = 0, sa = 0;
    for (int m = 0; m < nmol; ++m) {
        if (nbf_per_mol[m] < 1 || natom_per_mol[m] < 0) return fail(MMD_ERR_ARG, "molecule %d is empty", m);
        sf += nbf_per_mol[m];
        sa += natom_per_mol[m];
    }
    if (sf != ctx->nbf) return fail(MMD_ERR_ARG, "molecule sizes add up to %lld functions, the basis has %d",
                                    (long long)sf, ctx->nbf);
    if (sa != ctx->natom) return fail(MMD_ERR_ARG, "molecule atom counts add up to %lld, %d atoms are set",
                                      (long long)sa, ctx->natom);
    ctx->nmol = nmol;
    ctx->mol_f0.assign(nmol, 0);
    ctx->mol_n.assign(nmol, 0);
    ctx->rw = 0;
    std::vector<int2> pl;
    for (int m = 0, f = 0; m < nmol; ++m) {
        ctx->mol_f0[m] = f;
        ctx->mol_n[m] = nbf_per_mol[m];
        ctx->rw = std::max(ctx->rw, nbf_per_mol[m]);
        for (int i = f; i < f + nbf_per_mol[m]; ++i) {
            ctx->bf[i].pad = m;
            for (int j = f; j <= i; ++j) pl.push_back(make_int2(i, j));
        }
        f += nbf_per_mol[m];
    }
    ctx->mol_atoms.clear();
    for (int m = 0, a0 = 0; m < nmol; a0 += natom_per_mol[m], ++m) ctx->mol_atoms.push_back(make_int2(a0, natom_per_mol[m]));
    ctx->npl = (int64_t)pl.size();
    HIP_TRY(hipMemcpyAsync(ctx->d_bf.p, ctx->bf.data(), sizeof(BFDesc) * ctx->nbf, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(ctx->d_plist.reserve(pl.size()));
    HIP_TRY(hipMemcpyAsync(ctx->d_plist.p, pl.data(), sizeof(int2) * pl.size(), hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(ctx->d_mol_atoms.reserve(ctx->mol_atoms.size()));
    HIP_TRY(hipMemcpyAsync(ctx->d_mol_atoms.p, ctx->mol_atoms.data(), sizeof(int2) * ctx->mol_atoms.size(),
                           hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    build_shells(ctx);
    if (ctx->shells_ok) {
        rc = upload_shells(ctx);
        if (rc) return rc;
    }
    ctx->pairs_ok = false;
    ctx->schwarz_ok = false;
    ctx->units_ok = false;
    return MMD_OK;
}

namespace {
// Bra slices and flat ket lists of the gradient's class kernels, from the
// pair table.
int build_grad_plan(mmd_ctx* c)
{
    if (c->grad_plan_ok) return MMD_OK;
    std::vector<ShellPair> pairs((size_t)c->pc_off[NPAIRCLASS]);
    HIP_TRY(hipMemcpyAsync(pairs.data(), c->d_pairs.p, sizeof(ShellPair) * pairs.size(), hipMemcpyDeviceToHost, c->st));
    HIP_TRY(hipStreamSynchronize(c->st));
    std::vector<int4> sl, one;
    std::vector<int2> flat;
    for (int pc = 0; pc < NPAIRCLASS; ++pc) {
        c->g_slice_off[pc] = (int)sl.size();
        c->g_one_off[pc] = (int)one.size();
        c->g_flat_off[pc] = (int)flat.size();
        // bra slices of grad_pslice primitive pairs, shorter where the whole
        // molecule would not give the class some 1000 work units: a slice is
        // a serial chain in every lane, and a small molecule leaves most of
        // the GPU idle ((H2O) cc-pVDZ, (pp|pp): 133 us in 10 workgroups of 16)
        int64_t kets = 0;
        for (int k = 0; k <= pc; ++k) kets += c->pc_npp[k];
        const int64_t prims = c->pc_npp[pc];
        int step = grad_pslice(pc);
        while (step > 1 && (prims / step) * (kets / 256 + 1) < 1024) step /= 2;
        for (int P = c->pc_off[pc]; P < c->pc_off[pc + 1]; ++P) {
            const int npp = pairs[P].npp;
            for (int i = 0; i < npp; ++i) flat.push_back(make_int2(P, i));
            const int end = (int)flat.size() - c->g_flat_off[pc];
            for (int i = 0; i < npp; i += step) sl.push_back(make_int4(P, i, std::min(npp, i + step), end));
            if (pc >= 4)   // (dp) and (dd): the bras of those classes
                for (int i = 0; i < npp; ++i) one.push_back(make_int4(P, i, i + 1, end));
        }
    }
    c->g_slice_off[NPAIRCLASS] = (int)sl.size();
    c->g_one_off[NPAIRCLASS] = (int)one.size();
    c->g_flat_off[NPAIRCLASS] = (int)flat.size();
    for (int pc = 0; pc <= NPAIRCLASS; ++pc) c->g_one_off[pc] += (int)sl.size();
    sl.insert(sl.end(), one.begin(), one.end());
    HIP_TRY(c->g_slices.reserve(std::max<size_t>(1, sl.size())));
    HIP_TRY(c->g_flat.reserve(std::max<size_t>(1, flat.size())));
    HIP_TRY(hipMemcpyAsync(c->g_slices.p, sl.data(), sizeof(int4) * sl.size(), hipMemcpyHostToDevice, c->st));
    HIP_TRY(hipMemcpyAsync(c->g_flat.p, flat.data(), sizeof(int2) * flat.size(), hipMemcpyHostToDevice, c->st));
    HIP_TRY(hipStreamSynchronize(c->st));
    c->grad_plan_ok = true;
    return MMD_OK;
}

// The gradient by shell class: the one-electron pair classes and the 21
// quartet classes, spread over the context's streams by their work.
int gradient_shells(mmd_ctx* c, const double* dP, const double* dW, const double* nuc, double* dg)
{
    int rc;
    if (!c->pairs_ok && (rc = build_pairs(c, nullptr))) return rc;
    if ((rc = onee_pair_list(c))) return rc;
    if ((rc = build_grad_plan(c))) return rc;
    const size_t nrep = (size_t)GRAD_REPLICAS * 3 * c->natom;
    HIP_TRY(c->g_rep.reserve(nrep));
    HIP_TRY(launch_fill(nrep, c->g_rep.p, 0.0, c->st));
    GradArgs A;
    A.pairs = c->d_pairs.p;
    A.pp = c->d_pp.p;
    A.ppa = c->d_ppa.p;
    A.boys = c->d_boys.p;
    A.gcomp = c->d_gcomp.p;
    A.P = dP;
    A.bf_atom = c->g_atom.p;
    A.grad = c->g_rep.p;
    A.N = c->nbf;
    A.natom = c->natom;
    A.lds_atoms = c->natom <= 256 ? 1 : 0;   // 6 KB of LDS at most beside the class's own
    std::vector<StreamTask> tasks;   // quartet classes, then (from NQCLASS) one-electron pair classes
    GradClass cls[NQCLASS];
    for (int qc = 0; qc < NQCLASS; ++qc) {
        int pcb, pck, la, lb, lc, ld;
        class_of(qc, &pcb, &pck);
        qclass_decode(qc, &la, &lb, &lc, &ld);
        const bool block = fock_class_is_mfma(la, lb, lc, ld);   // a workgroup per primitive quartet
        const int* off = block ? c->g_one_off : c->g_slice_off;
        GradClass& C = cls[qc];
        C.slices = c->g_slices.p + off[pcb];
        C.nslice = off[pcb + 1] - off[pcb];
        C.flat = c->g_flat.p + c->g_flat_off[pck];
        C.nflat = c->g_flat_off[pck + 1] - c->g_flat_off[pck];
        C.nkc = (C.nflat + 255) / 256;
        C.tri = pcb == pck ? 1 : 0;
        if (C.nslice == 0 || C.nflat == 0) continue;
        const double prims = (double)(c->g_flat_off[pcb + 1] - c->g_flat_off[pcb]) * C.nflat * (C.tri ? 0.5 : 1.0);
        const double work = 100.0 + nherm(la + lb + lc + ld + 1) * 6.0
                          + 3.0 * ncart(la) * ncart(lb) * nherm(la + lb) * nherm(lc + ld);
        tasks.push_back({prims * work + 1e6, qc});   // 1e6: a launch's fixed latency
    }
    OneeArgs O = onee_args(c);
    for (int pc = 0; pc < NPAIRCLASS; ++pc)
        if (c->onee_off[pc + 1] > c->onee_off[pc])
            tasks.push_back({1e6 + 1e4 * (c->onee_off[pc + 1] - c->onee_off[pc]), NQCLASS + pc});
    rc = spread_tasks(c, tasks, [&](int id, hipStream_t sq) {
        if (id < NQCLASS) return launch_grad_class(id, A, cls[id], sq);
        const int pc = id - NQCLASS;
        return launch_grad_onee(pc, O, c->d_onee_list.p + c->onee_off[pc], c->onee_off[pc + 1] - c->onee_off[pc],
                                c->g_atom.p, dP, dW, c->g_rep.p, sq);
    });
    if (rc) return rc;
    HIP_TRY(launch_grad_sum(c->natom, GRAD_REPLICAS, c->g_rep.p, nuc, dg, c->st));
    return MMD_OK;
}
}  // namespace

namespace {
int rhf_gradient(mmd_ctx* ctx, const double* P, const double* W, const int32_t* bf_atom, const double* nuc,
                 double* grad)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    const int N = ctx->nbf, natom = ctx->natom;
    if (N == 0) return fail(MMD_ERR_STATE, "no basis set");
    if (natom < 1) return fail(MMD_ERR_STATE, "no nuclei (mmd_set_atoms)");
    if (ctx->nmol > 1) return fail(MMD_ERR_UNSUPPORTED, "the gradient takes one molecule, not a batch");
    if (natom > 4096) return fail(MMD_ERR_UNSUPPORTED, "the gradient takes up to 4096 atoms");
    if (!P || !W || !bf_atom || !grad) return fail(MMD_ERR_ARG, "null pointer");
    for (int i = 0; i < N; ++i)
        if (bf_atom[i] < 0 || bf_atom[i] >= natom) return fail(MMD_ERR_ARG, "basis function %d: atom out of range", i);
    const size_t nn = (size_t)N * N;
    HIP_TRY(ctx->g_PW.reserve(2 * nn + 7 * (size_t)natom));
    HIP_TRY(ctx->g_atom.reserve(N));
    double* dP = ctx->g_PW.p;
    double* dW = dP + nn;
    double* dg = dW + nn;
    double* dn = nuc ? dg + 3 * (size_t)natom : nullptr;
    HIP_TRY(hipMemcpyAsync(dP, P, sizeof(double) * nn, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(dW, W, sizeof(double) * nn, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(ctx->g_atom.p, bf_atom, sizeof(int32_t) * N, hipMemcpyHostToDevice, ctx->st));
    if (nuc) HIP_TRY(hipMemcpyAsync(dn, nuc, sizeof(double) * 4 * natom, hipMemcpyHostToDevice, ctx->st));
    // whole shells, each on one atom: the shell-class kernels; else the
    // per-function kernels
    bool shells = ctx->shells_ok;
    for (size_t k = 0; k < ctx->shells.size() && shells; ++k)
        for (int i = 1; i < ncart(ctx->shells[k].l); ++i)
            shells = shells && bf_atom[ctx->shells[k].bf0 + i] == bf_atom[ctx->shells[k].bf0];
    HIP_TRY(hipEventRecord(ctx->ev0, ctx->st));
    if (shells) {
        if ((rc = gradient_shells(ctx, dP, dW, dn, dg))) return rc;
    } else {
        HIP_TRY(launch_fill(3 * (size_t)natom, dg, 0.0, ctx->st));
        HIP_TRY(launch_rhf_gradient(N, ctx->d_bf.p, ctx->d_bf_exp.p, ctx->d_bf_w.p, natom, ctx->d_atoms.p,
                                    ctx->d_boys.p, ctx->g_atom.p, dP, dW, dg, ctx->st));
        if (dn) HIP_TRY(launch_grad_sum(natom, 1, dg, dn, dg, ctx->st));
    }
    HIP_TRY(hipEventRecord(ctx->ev1, ctx->st));
    HIP_TRY(hipMemcpyAsync(grad, dg, sizeof(double) * 3 * natom, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    ctx->last_grad_ms = ms;
    return MMD_OK;
}

}  // namespace

int mmd_rhf_gradient(mmd_ctx* ctx, const double* P, const double* W, const int32_t* bf_atom, double* grad)
{
    return rhf_gradient(ctx, P, W, bf_atom, nullptr, grad);
}

int mmd_rhf_total_gradient(mmd_ctx* ctx, const double* P, const double* W, const int32_t* bf_atom,
                           const double* nuclei, double* grad)
{
    if (!nuclei) return fail(MMD_ERR_ARG, "null pointer");
    return rhf_gradient(ctx, P, W, bf_atom, nuclei, grad);
}

int mmd_last_gradient_ms(mmd_ctx* ctx, double* ms)
{
    if (!ctx || !ms) return fail(MMD_ERR_ARG, "null pointer");
    *ms = ctx->last_grad_ms;
    return MMD_OK;
}

int mmd_one_electron(mmd_ctx* ctx, const double center[3], double* S, double* T, double* V, double* M, double* L)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (ctx->nbf == 0) return fail(MMD_ERR_STATE, "no basis set");
    if (!center || !S || !T || !V || !M || !L) return fail(MMD_ERR_ARG, "null pointer");
    const size_t nn = (size_t)ctx->nbf * ctx->nbf;
    DevBuf<double>& d = ctx->d_onee;   // kept between calls (no allocation per SCF)
    HIP_TRY(d.reserve(9 * nn));
    const bool several = ctx->nmol > 1;
    if (ctx->shells_ok) {
        if ((rc = one_electron_shells(ctx, center, d.p, d.p + nn, d.p + 2 * nn, d.p + 3 * nn, d.p + 6 * nn)))
            return rc;
    } else {
        HIP_TRY(launch_one_electron(ctx->nbf, ctx->d_bf.p, ctx->d_bf_exp.p, ctx->d_bf_w.p, ctx->natom,
                                    ctx->natom ? ctx->d_atoms.p : nullptr, center[0], center[1], center[2],
                                    ctx->d_boys.p, d.p, d.p + nn, d.p + 2 * nn, d.p + 3 * nn, d.p + 6 * nn, ctx->st,
                                    several ? ctx->d_plist.p : nullptr, ctx->npl,
                                    several ? ctx->d_mol_atoms.p : nullptr));
    }
    HIP_TRY(hipMemcpyAsync(S, d.p, sizeof(double) * nn, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipMemcpyAsync(T, d.p + nn, sizeof(double) * nn, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipMemcpyAsync(V, d.p + 2 * nn, sizeof(double) * nn, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipMemcpyAsync(M, d.p + 3 * nn, sizeof(double) * 3 * nn, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipMemcpyAsync(L, d.p + 6 * nn, sizeof(double) * 3 * nn, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    return MMD_OK;
}

int mmd_schwarz(mmd_ctx* ctx, double* diag)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (ctx->nbf == 0) return fail(MMD_ERR_STATE, "no basis set");
    const int N = ctx->nbf;
    const size_t nn = (size_t)N * N;
    HIP_TRY(ctx->d_schwarz.reserve(nn));
    if ((rc = schwarz_diagonal(ctx, ctx->d_schwarz.p))) return rc;
    if (diag) HIP_TRY(hipMemcpyAsync(diag, ctx->d_schwarz.p, sizeof(double) * nn, hipMemcpyDeviceToHost, ctx->st));
    return finish_schwarz(ctx);
}

int mmd_set_schwarz(mmd_ctx* ctx, const double* diag)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (ctx->nbf == 0) return fail(MMD_ERR_STATE, "no basis set");
    if (!diag) return fail(MMD_ERR_ARG, "null pointer");
    const size_t nn = (size_t)ctx->nbf * ctx->nbf;
    HIP_TRY(ctx->d_schwarz.reserve(nn));
    HIP_TRY(hipMemcpyAsync(ctx->d_schwarz.p, diag, sizeof(double) * nn, hipMemcpyHostToDevice, ctx->st));
    return finish_schwarz(ctx);
}

namespace {
// Staged bra data of every pair class, from the pair table.
int build_bra_tables(mmd_ctx* c)
{
    if (c->btab_ok) return MMD_OK;
    size_t total = 0;
    for (int pc = 0; pc < NPAIRCLASS; ++pc) {
        c->btab_off[pc] = total;
        total += (size_t)c->pc_npp[pc] * bra_table_stride(pc);
    }
    HIP_TRY(c->d_btab.reserve(std::max<size_t>(1, total)));
    for (int pc = 0; pc < NPAIRCLASS; ++pc)
        HIP_TRY(launch_bra_table(pc, c->d_pairs.p, c->d_pp.p, c->pc_off[pc], c->pc_off[pc + 1] - c->pc_off[pc],
                                 c->d_btab.p + c->btab_off[pc], c->st));
    c->btab_ok = true;
    return MMD_OK;
}

// Every quartet class on the integral-block kernels (the stored tensor, or a
// raw build with the fields of `raw`), side by side on the context's streams.
int run_block_classes(mmd_ctx* c, const ClassArgs& A, const BlockArgs& raw)
{
    if (int rc = build_bra_tables(c)) return rc;
    std::vector<StreamTask> tasks;
    BlockArgs cls[NQCLASS];
    const int* npp = c->pc_npp;
    for (int qc = 0; qc < NQCLASS; ++qc) {
        int pcb, pck, la, lb, lc, ld;
        class_of(qc, &pcb, &pck);
        qclass_decode(qc, &la, &lb, &lc, &ld);
        BlockArgs& B = cls[qc];
        B = raw;
        B.boff = c->pc_off[pcb];
        B.nb = c->pc_off[pcb + 1] - B.boff;
        B.koff = c->pc_off[pck];
        B.nk = c->pc_off[pck + 1] - B.koff;
        B.tri = pcb == pck ? 1 : 0;
        B.table = c->d_btab.p + c->btab_off[pcb];
        if (B.nb == 0 || B.nk == 0) continue;
        // lanes per quartet from the classes' mean contraction lengths, at
        // least four (the LDS blocks of a wavefront hold sixteen groups)
        auto lg = [](int64_t n, int64_t pairs) { return n >= 3 * pairs ? 2 : (2 * n >= 3 * pairs ? 1 : 0); };
        B.lgb = lg(npp[pcb], B.nb);
        B.lgk = lg(npp[pck], B.nk);
        if (B.lgb + B.lgk < 2) B.lgk = 2 - B.lgb;
        const double prims = (double)npp[pcb] * npp[pck] * (B.tri ? 0.5 : 1.0);
        tasks.push_back({1e6 + prims * (40.0 + 4.0 * nherm(la + lb + lc + ld)
                                        + (double)ncart(la) * ncart(lb) * ncart(lc) * ncart(ld)), qc});
    }
    return spread_tasks(c, tasks, [&](int qc, hipStream_t sq) { return launch_block_class(qc, A, cls[qc], sq); });
}

// The full (ij|kl) tensor from the shell-pair tables: every quartet class
// with bra pair class >= ket pair class, all canonical shell quartets of it
// (bra pair >= ket pair inside one pair class), every integral stored at its
// eight index permutations.  Every element of dst is written.
int eri_tensor_shells(mmd_ctx* c, double* dst)
{
    ClassArgs A = base_args(c);
    A.G = dst;
    BlockArgs B;
    memset(&B, 0, sizeof(B));
    return run_block_classes(c, A, B);
}

// formPT's unsymmetrised G of the density difference in d_D (and d_Dim) with
// |dP| in d_absD, into d_graw: the real matrix, then the imaginary one.
int raw_fock_shells(mmd_ctx* c, bool complex_dP, double tol)
{
    const size_t nn = (size_t)c->nbf * c->nbf;
    HIP_TRY(launch_shell_block_max_raw((int)c->shells.size(), c->d_sh_bf0.p, c->d_sh_nbf.p, c->nbf, c->d_absD.p,
                                       c->d_Dsh.p, c->st));
    if (!c->qraw_ok) {   // from the pair table and the Schwarz diagonal, which rebuilds it
        const int n = c->pc_off[NPAIRCLASS];
        HIP_TRY(c->d_qraw.reserve((size_t)n));
        HIP_TRY(launch_pair_qraw(n, c->d_pairs.p, c->d_sh_nbf.p, c->nbf, c->d_sqS.p, c->d_qraw.p, c->st));
        c->qraw_ok = true;
    }
    // copies of G, so that the updates of a small matrix do not queue at the
    // same addresses; 128 MB of them at most
    const int nrep = (int)std::max<size_t>(1, std::min<size_t>(16, (size_t(8) << 20) / nn));
    HIP_TRY(c->d_graw.reserve(nrep * 2 * nn));
    HIP_TRY(launch_fill(nrep * 2 * nn, c->d_graw.p, 0.0, c->st));
    ClassArgs A = base_args(c);
    A.D = c->d_D.p;
    A.absD = c->d_absD.p;
    A.sqS = c->d_sqS.p;
    A.tol = tol;
    A.G = c->d_graw.p;
    BlockArgs B;
    memset(&B, 0, sizeof(B));
    B.raw = 1;
    B.nrep = nrep;
    B.Dim = complex_dP ? c->d_Dim.p : nullptr;
    B.Dsh = c->d_Dsh.p;
    B.qraw = c->d_qraw.p;
    B.nshell = (int)c->shells.size();
    if (int rc = run_block_classes(c, A, B)) return rc;
    HIP_TRY(launch_sum_copies((complex_dP ? 2 : 1) * nn, nrep, 2 * nn, c->d_graw.p, c->d_graw.p, c->st));
    return MMD_OK;
}
}  // namespace

int mmd_eri_tensor(mmd_ctx* ctx, double* out, int out_on_device)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (!out) return fail(MMD_ERR_ARG, "null output");
    if (ctx->nbf == 0) return fail(MMD_ERR_STATE, "no basis set");
    const size_t n4 = (size_t)ctx->nbf * ctx->nbf * ctx->nbf * ctx->nbf;
    Tensor4 t;
    HostStage stage;
    double* dst = out;
    if (!out_on_device) {
        HIP_TRY(t.reserve(n4));
        dst = t.p;
    }
    if (ctx->shells_ok) {
        if (!ctx->pairs_ok) {
            rc = build_pairs(ctx, nullptr);
            if (rc) return rc;
        }
        if ((rc = eri_tensor_shells(ctx, dst))) return rc;
    } else {
        HIP_TRY(launch_canonical_quartets(0, ctx->nbf, ctx->d_bf.p, ctx->d_bf_exp.p, ctx->d_bf_w.p, ctx->d_boys.p,
                                          nullptr, nullptr, nullptr, 0.0, dst, ctx->st));
    }
    if (!out_on_device) HIP_TRY(stage.to_host(out, dst, sizeof(double) * n4, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    t.done();
    return MMD_OK;
}

int mmd_eri_list(mmd_ctx* ctx, int64_t n, const int64_t* ijkl, double* out)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (ctx->nbf == 0) return fail(MMD_ERR_STATE, "no basis set");
    if (n < 0 || (n > 0 && (!ijkl || !out))) return fail(MMD_ERR_ARG, "invalid quartet list");
    if (n == 0) return MMD_OK;
    for (int64_t i = 0; i < 4 * n; ++i)
        if (ijkl[i] < 0 || ijkl[i] >= ctx->nbf) return fail(MMD_ERR_ARG, "basis-function index out of range");
    DevBuf<int64_t> d_idx;
    DevBuf<double> d_out;
    HIP_TRY(d_idx.reserve(4 * n));
    HIP_TRY(d_out.reserve(n));
    HIP_TRY(hipMemcpyAsync(d_idx.p, ijkl, sizeof(int64_t) * 4 * n, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(launch_eri_bf_list(n, d_idx.p, ctx->d_bf.p, ctx->d_bf_exp.p, ctx->d_bf_w.p, ctx->d_boys.p, d_out.p, ctx->st));
    HIP_TRY(hipMemcpyAsync(out, d_out.p, sizeof(double) * n, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    return MMD_OK;
}

int mmd_fock_delta(mmd_ctx* ctx, const double* dP_re, const double* dP_im, double tol, int raw, double* G_re,
                   double* G_im, int on_device, int64_t* nsurv)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (!ctx->schwarz_ok) return fail(MMD_ERR_STATE, "mmd_schwarz must be called before mmd_fock_delta");
    if (!dP_re || !G_re || (dP_im && !G_im)) return fail(MMD_ERR_ARG, "null pointer");
    if (!raw && dP_im) return fail(MMD_ERR_ARG, "the symmetrised build needs a real density difference");
    if (!raw && !ctx->pairs_ok) return fail(MMD_ERR_UNSUPPORTED, "%s", ctx->shells_err.c_str());
    const int N = ctx->nbf;
    const size_t nn = (size_t)N * N;
    const hipMemcpyKind k_in = on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    const hipMemcpyKind k_out = on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost;
    HIP_TRY(hipEventRecord(ctx->ev0, ctx->st));
    HIP_TRY(hipMemcpyAsync(ctx->d_D.p, dP_re, sizeof(double) * nn, k_in, ctx->st));
    if (dP_im) HIP_TRY(hipMemcpyAsync(ctx->d_Dim.p, dP_im, sizeof(double) * nn, k_in, ctx->st));
    if (raw)
        HIP_TRY(launch_abs_density((int)nn, ctx->d_D.p, dP_im ? ctx->d_Dim.p : nullptr, ctx->d_absD.p, ctx->st));
    if (!raw) {
        HIP_TRY(launch_fock_prep(N, ctx->d_D.p, ctx->d_absD.p, ctx->d_G.p, ctx->d_sh_bf0.p, ctx->d_sh_nbf.p,
                                 (int)ctx->shells.size(), ctx->d_Dsh.p, reinterpret_cast<int*>(ctx->d_ctr.p),
                                 FOCK_COUNTER_WORDS, ctx->st));
        ClassArgs A = base_args(ctx);
        A.absD = ctx->d_absD.p;
        A.sqS = ctx->d_sqS.p;
        A.tol = tol;
        A.D = ctx->d_D.p;
        A.G = ctx->d_G.p;
        FockScratch W;
        W.counters(ctx->d_ctr.p);
        W.Dsh = ctx->d_Dsh.p;
        rc = run_fock_classes(ctx, A, tol, W);
        if (rc) return rc;
        HIP_TRY(launch_symmetrize(N, ctx->d_G.p, ctx->d_Gout.p, ctx->st, reinterpret_cast<const int*>(ctx->d_ctr.p),
                                  reinterpret_cast<int*>(ctx->h_ctr), FOCK_REPORT_WORDS));
        HIP_TRY(hipMemcpyAsync(G_re, ctx->d_Gout.p, sizeof(double) * nn, k_out, ctx->st));
    } else if (ctx->pairs_ok && ctx->nmol == 1) {
        if ((rc = raw_fock_shells(ctx, dP_im != nullptr, tol))) return rc;
        HIP_TRY(hipMemcpyAsync(G_re, ctx->d_graw.p, sizeof(double) * nn, k_out, ctx->st));
        if (dP_im) HIP_TRY(hipMemcpyAsync(G_im, ctx->d_graw.p + nn, sizeof(double) * nn, k_out, ctx->st));
    } else {   // functions that do not form whole shells, or several molecules
        for (int part = 0; part < (dP_im ? 2 : 1); ++part) {
            HIP_TRY(launch_fill(nn, ctx->d_G.p, 0.0, ctx->st));
            HIP_TRY(launch_canonical_quartets(1, N, ctx->d_bf.p, ctx->d_bf_exp.p, ctx->d_bf_w.p, ctx->d_boys.p,
                                              part == 0 ? ctx->d_D.p : ctx->d_Dim.p, ctx->d_absD.p, ctx->d_sqS.p, tol,
                                              ctx->d_G.p, ctx->st));
            HIP_TRY(hipMemcpyAsync(part == 0 ? G_re : G_im, ctx->d_G.p, sizeof(double) * nn, k_out, ctx->st));
        }
    }
    HIP_TRY(hipEventRecord(ctx->ev1, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    if (!raw) count_survivors(ctx);
    if (nsurv) *nsurv = raw ? -1 : ctx->last_nsurv;
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    ctx->last_fock_ms = ms;
    if (!raw && ctx->plan_measuring) {
        for (int qc = 0; qc < NQCLASS; ++qc) {
            float cms = 0.f;
            if (ctx->qc_total[qc]) HIP_TRY(hipEventElapsedTime(&cms, ctx->evc[3 * qc], ctx->evc[3 * qc + 2]));
            ctx->plan_ms[qc] = cms > 0.f ? cms : 1e-3;
        }
        ctx->plan_measuring = false;
        ctx->plan_countdown = mmd_ctx::PLAN_EVERY;
    } else if (!raw) {
        --ctx->plan_countdown;
    }
    if (!raw && ctx->tune_measuring) {
        // a build of the implementation choice: record, and decide after both
        for (int qc = 0; qc < NQCLASS; ++qc) {
            float cms = 0.f;
            if (ctx->qc_total[qc]) HIP_TRY(hipEventElapsedTime(&cms, ctx->evc[3 * qc], ctx->evc[3 * qc + 2]));
            ctx->tune_ms[ctx->tune_phase][qc] = cms;
        }
        ctx->tune_measuring = false;
        if (++ctx->tune_phase == 2) {
            for (int qc = 0; qc < NQCLASS; ++qc) {
                int la, lb, lc, ld;
                qclass_decode(qc, &la, &lb, &lc, &ld);
                if (fock_class_has_both(la, lb, lc, ld))
                    ctx->impl_choice[qc] = ctx->tune_ms[1][qc] < ctx->tune_ms[0][qc] ? 1 : 0;
            }
            ctx->plan_countdown = 0;   // plan again on the chosen kernels
        }
    }
    if (ctx->profiling && !raw) return collect_profile(ctx);
    return MMD_OK;
}

// The symmetrised build of mmd_fock_delta (raw = 0, real dP, device
// pointers) with every work buffer in the static `scratch` of this device
// instead of the context's: |dP|, the shell-block maxima, the unsymmetrised
// accumulator, counters and survivor lists.  No allocation on the host or the
// device; the kernels are the same.
int mmd_fock_delta_noalloc(mmd_ctx* ctx, const double* dP, double tol, double* G, int64_t* nsurv)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (!ctx->schwarz_ok) return fail(MMD_ERR_STATE, "mmd_schwarz must be called before mmd_fock_delta_noalloc");
    if (!ctx->pairs_ok) return fail(MMD_ERR_UNSUPPORTED, "%s", ctx->shells_err.c_str());
    if (!ctx->units_ok) return fail(MMD_ERR_STATE, "work units missing (set the Schwarz screen again)");
    if (!dP || !G) return fail(MMD_ERR_ARG, "null pointer");
    if (!ctx->noalloc_scratch) return fail(MMD_ERR_STATE, "no scratch address for this device");
    const int N = ctx->nbf;
    const size_t nn = (size_t)N * N;
    const size_t ns = ctx->shells.size();
    auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
    unsigned char* base = static_cast<unsigned char*>(ctx->noalloc_scratch);
    size_t off = 0;
    double* absD = reinterpret_cast<double*>(base + off);
    off += up(sizeof(double) * nn);
    double* Gacc = reinterpret_cast<double*>(base + off);
    off += up(sizeof(double) * nn);
    double* Dsh = reinterpret_cast<double*>(base + off);
    off += up(sizeof(double) * ns * ns);
    FockCounters* ctr = ctx->d_ctr.p;   // allocated with the tables
    if (off > NOALLOC_SCRATCH_BYTES)
        return fail(MMD_ERR_ARG, "a basis of %d functions needs %zu bytes of scratch; the limit is %zu", N, off,
                    NOALLOC_SCRATCH_BYTES);
    FockScratch W;
    W.counters(ctr);
    W.Dsh = Dsh;
    W.surv = reinterpret_cast<int2*>(base + off);
    W.surv_cap = (int64_t)((NOALLOC_SCRATCH_BYTES - off) / sizeof(int2));
    W.allow_measure = false;
    HIP_TRY(hipEventRecord(ctx->ev0, ctx->st));
    HIP_TRY(launch_fock_prep(N, dP, absD, Gacc, ctx->d_sh_bf0.p, ctx->d_sh_nbf.p, (int)ns, Dsh,
                             reinterpret_cast<int*>(ctr), FOCK_COUNTER_WORDS, ctx->st));
    ClassArgs A = base_args(ctx);
    A.absD = absD;
    A.sqS = ctx->d_sqS.p;
    A.tol = tol;
    A.D = dP;
    A.G = Gacc;
    rc = run_fock_classes(ctx, A, tol, W);
    if (rc) return rc;
    HIP_TRY(launch_symmetrize(N, Gacc, G, ctx->st, reinterpret_cast<const int*>(ctr),
                              reinterpret_cast<int*>(ctx->h_ctr), FOCK_REPORT_WORDS));
    HIP_TRY(hipEventRecord(ctx->ev1, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    count_survivors(ctx);
    if (nsurv) *nsurv = ctx->last_nsurv;
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    ctx->last_fock_ms = ms;
    return MMD_OK;
}

int mmd_jk_tensor(mmd_ctx* ctx, const double* T, int t_on_device, const double* P_re, const double* P_im,
                  double* J_re, double* J_im, double* K_re, double* K_im)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (ctx->nbf == 0) return fail(MMD_ERR_STATE, "no basis set");
    if (!T || !P_re || !J_re || !K_re || (P_im && (!J_im || !K_im))) return fail(MMD_ERR_ARG, "null pointer");
    const int N = ctx->nbf;
    const size_t nn = (size_t)N * N, n4 = nn * nn;
    Tensor4 dT;
    HostStage stage;
    DevBuf<double>& d = ctx->jk_mats;
    const double* t = T;
    if (!t_on_device) {
        HIP_TRY(dT.reserve(n4));
        HIP_TRY(stage.to_device(dT.p, T, sizeof(double) * n4, ctx->st));
        t = dT.p;
    }
    HIP_TRY(d.reserve(6 * nn));
    HIP_TRY(hipMemcpyAsync(d.p, P_re, sizeof(double) * nn, hipMemcpyHostToDevice, ctx->st));
    if (P_im) HIP_TRY(hipMemcpyAsync(d.p + nn, P_im, sizeof(double) * nn, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(launch_jk_tensor(N, t, d.p, P_im ? d.p + nn : nullptr, d.p + 2 * nn, d.p + 3 * nn, d.p + 4 * nn,
                             d.p + 5 * nn, ctx->st));
    HIP_TRY(hipMemcpyAsync(J_re, d.p + 2 * nn, sizeof(double) * nn, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipMemcpyAsync(K_re, d.p + 4 * nn, sizeof(double) * nn, hipMemcpyDeviceToHost, ctx->st));
    if (P_im) {
        HIP_TRY(hipMemcpyAsync(J_im, d.p + 3 * nn, sizeof(double) * nn, hipMemcpyDeviceToHost, ctx->st));
        HIP_TRY(hipMemcpyAsync(K_im, d.p + 5 * nn, sizeof(double) * nn, hipMemcpyDeviceToHost, ctx->st));
    }
    HIP_TRY(hipStreamSynchronize(ctx->st));
    dT.done();
    stage.done();
    return MMD_OK;
}

int mmd_boys(mmd_ctx* ctx, int n, const double* m, const double* T, int table, double* out)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (n < 0 || (n > 0 && (!m || !T || !out))) return fail(MMD_ERR_ARG, "invalid arguments");
    for (int i = 0; i < n; ++i) {
        if (!(m[i] >= 0.0) || !(T[i] >= 0.0)) return fail(MMD_ERR_ARG, "Boys arguments must be non-negative");
        if (table && (m[i] != floor(m[i]) || m[i] > MAX_LTOT))
            return fail(MMD_ERR_ARG, "tabulated Boys path takes integer m <= %d", MAX_LTOT);
    }
    if (n == 0) return MMD_OK;
    DevBuf<double> d;
    HIP_TRY(d.reserve(3 * (size_t)n));
    HIP_TRY(hipMemcpyAsync(d.p, m, sizeof(double) * n, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(d.p + n, T, sizeof(double) * n, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(launch_boys_eval(n, d.p, d.p + n, table, ctx->d_boys.p, d.p + 2 * n, ctx->st));
    HIP_TRY(hipMemcpyAsync(out, d.p + 2 * n, sizeof(double) * n, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    return MMD_OK;
}

int mmd_set_profiling(mmd_ctx* ctx, int on)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (on && !ctx->evc[0])
        for (int i = 0; i < 3 * NQCLASS; ++i) HIP_TRY(hipEventCreate(&ctx->evc[i]));
    if (on)
        for (auto& a : ctx->psum) a = ProfileSum();
    if (on < 0 || on > 2) return fail(MMD_ERR_ARG, "profiling mode must be 0, 1 or 2");
    ctx->profiling = on;
    return MMD_OK;
}

int mmd_fock_stats(mmd_ctx* ctx, int32_t* lclass, int64_t* nquart, int64_t* nprim, double* ms)
{
    if (!ctx) return fail(MMD_ERR_ARG, "null context");
    for (int qc = 0; qc < NQCLASS; ++qc) {
        if (lclass) qclass_decode(qc, &lclass[4 * qc], &lclass[4 * qc + 1], &lclass[4 * qc + 2], &lclass[4 * qc + 3]);
        if (nquart) nquart[qc] = ctx->st_nquart[qc];
        if (nprim) nprim[qc] = ctx->st_nprim[qc];
        if (ms) ms[qc] = ctx->st_ms[qc];
    }
    return NQCLASS;
}

int mmd_fock_profile_sums(mmd_ctx* ctx, int32_t* lclass, int64_t* nquart, int64_t* nprim, double* ms,
                          int64_t* builds)
{
    if (!ctx) return fail(MMD_ERR_ARG, "null context");
    for (int qc = 0; qc < NQCLASS; ++qc) {
        const ProfileSum& a = ctx->psum[qc];
        if (lclass) qclass_decode(qc, &lclass[4 * qc], &lclass[4 * qc + 1], &lclass[4 * qc + 2], &lclass[4 * qc + 3]);
        for (int t = 0; t < 2; ++t) {
            if (nquart) nquart[2 * qc + t] = a.nquart[t];
            if (nprim) nprim[2 * qc + t] = a.nprim[t];
            if (ms) ms[2 * qc + t] = a.ms[t];
        }
        if (builds) builds[qc] = a.builds;
    }
    return NQCLASS;
}

int mmd_set_ket_slices(mmd_ctx* ctx, const int32_t* slices, int32_t* current)
{
    if (!ctx) return fail(MMD_ERR_ARG, "null context");
    if (slices) {
        for (int qc = 0; qc < NQCLASS; ++qc)
            if (slices[qc] != 0 && (slices[qc] < 1 || slices[qc] > KSLICE_MAX))
                return fail(MMD_ERR_ARG, "class %d: ket slice %d outside 1..%d", qc, (int)slices[qc], KSLICE_MAX);
        for (int qc = 0; qc < NQCLASS; ++qc)
            if (slices[qc] != 0) ctx->ket_slice[qc] = slices[qc];
    }
    if (current)
        for (int qc = 0; qc < NQCLASS; ++qc) current[qc] = ctx->ket_slice[qc];
    return MMD_OK;
}

int mmd_set_class_impl(mmd_ctx* ctx, int mode, int32_t* choice)
{
    if (!ctx) return fail(MMD_ERR_ARG, "null context");
    if (mode < -1 || mode > 2) return fail(MMD_ERR_ARG, "mode must be 0 (row), 1 (matrix cores), 2 (measured) or -1");
    if (mode >= 0 && mode != ctx->impl_mode) {
        ctx->impl_mode = mode;
        for (int qc = 0; qc < NQCLASS; ++qc) ctx->impl_choice[qc] = -1;
        ctx->tune_phase = 0;
        ctx->plan_countdown = 0;
    }
    if (choice)
        for (int qc = 0; qc < NQCLASS; ++qc) {
            int la, lb, lc, ld;
            qclass_decode(qc, &la, &lb, &lc, &ld);
            const bool both = fock_class_has_both(la, lb, lc, ld);
            const bool mf = fock_class_is_wave(la, lb, lc, ld);
            choice[qc] = !mf ? 0 : (!both ? 1 : (ctx->impl_mode == 2 ? ctx->impl_choice[qc] : ctx->impl_mode));
        }
    return MMD_OK;
}

int mmd_set_precision(mmd_ctx* ctx, double fp32_below)
{
    if (!ctx) return fail(MMD_ERR_ARG, "null context");
    if (!(fp32_below >= 0.0) || fp32_below > 1.0) return fail(MMD_ERR_ARG, "fp32_below must be in [0, 1]");
    ctx->fp32_below = fp32_below;
    return MMD_OK;
}

int mmd_set_streams(mmd_ctx* ctx, int n)
{
    if (!ctx) return fail(MMD_ERR_ARG, "null context");
    if (n < 1 || n > 1 + mmd_ctx::NSIDE) return fail(MMD_ERR_ARG, "streams must be in [1, %d]", 1 + mmd_ctx::NSIDE);
    if (ctx->nbf > 0) {
        HIP_TRY(hipSetDevice(ctx->device));
        if (int rc = ensure_streams(ctx, n)) return rc;
    }
    ctx->nstreams = n;
    return MMD_OK;
}

int mmd_set_lds_limit(mmd_ctx* ctx, int64_t bytes)
{
    if (!ctx) return fail(MMD_ERR_ARG, "null context");
    if (bytes < 0) return fail(MMD_ERR_ARG, "LDS limit must be >= 0");
    ctx->max_lds = bytes == 0 ? ctx->max_lds_device : std::min<size_t>((size_t)bytes, ctx->max_lds_device);
    return MMD_OK;
}

int mmd_fock_tiers(mmd_ctx* ctx, int64_t* nquart, int64_t* nquart_fp32)
{
    if (!ctx) return fail(MMD_ERR_ARG, "null context");
    if (nquart) *nquart = ctx->last_nsurv;
    if (nquart_fp32) *nquart_fp32 = ctx->last_nsurv_fp32;
    return MMD_OK;
}

}  // extern "C"

namespace {

// Row-major C (m x n) = op(A) op(B), op = transpose where tA / tB; the
// column-major BLAS computes C^T = op(B)^T op(A)^T.
int gemm_rm(mmd_ctx* c, bool tA, bool tB, int m, int n, int k, const double* A, int lda, const double* B, int ldb,
            double* C, int ldc)
{
    const double one = 1.0, zero = 0.0;
    const rocblas_status s = rocblas_dgemm(c->blas, tB ? rocblas_operation_transpose : rocblas_operation_none,
                                           tA ? rocblas_operation_transpose : rocblas_operation_none, n, m, k, &one,
                                           B, ldb, A, lda, &zero, C, ldc);
    if (s != rocblas_status_success) return fail(MMD_ERR_DEVICE, "rocblas_dgemm: status %d", (int)s);
    return MMD_OK;
}

// Solve the (n x n) system A x = b in place (Gaussian elimination with
// partial pivoting); false if singular.
bool solve_small(int n, std::vector<double>& A, std::vector<double>& b)
{
    for (int k = 0; k < n; ++k) {
        int piv = k;
        for (int i = k + 1; i < n; ++i)
            if (fabs(A[i * n + k]) > fabs(A[piv * n + k])) piv = i;
        if (A[piv * n + k] == 0.0) return false;
        if (piv != k) {
            for (int j = 0; j < n; ++j) std::swap(A[k * n + j], A[piv * n + j]);
            std::swap(b[k], b[piv]);
        }
        for (int i = k + 1; i < n; ++i) {
            const double f = A[i * n + k] / A[k * n + k];
            for (int j = k; j < n; ++j) A[i * n + j] -= f * A[k * n + j];
            b[i] -= f * b[k];
        }
    }
    for (int k = n - 1; k >= 0; --k) {
        double v = b[k];
        for (int j = k + 1; j < n; ++j) v -= A[k * n + j] * b[j];
        b[k] = v / A[k * n + k];
    }
    return true;
}

int scf_check(mmd_ctx* c)
{
    if (c->scf_n == 0 || c->scf_n != c->nbf) return fail(MMD_ERR_STATE, "mmd_scf_begin must be called first");
    return MMD_OK;
}

}  // namespace

extern "C" {

namespace {
// Enqueue G = sym(G(dP)) (the symmetrised build of mmd_fock_delta) on the
// context's stream: no allocation and no host synchronisation, so that a
// batched iteration can be captured into a graph.
int enqueue_fock_sym(mmd_ctx* c, const double* dP, double tol, double* Gout)
{
    const int N = c->nbf;
    const size_t nn = (size_t)N * N;
    const bool blocks = c->nmol > 1;   // a batch: only the molecules' diagonal blocks are live
    if (blocks) {
        HIP_TRY(launch_block_prep(c->nmol, c->d_mol_blocks.p, N, dP, c->d_absD.p, c->d_G.p, c->d_sh_bf0.p,
                                  c->d_sh_nbf.p, (int)c->shells.size(), c->d_Dsh.p, c->d_mol_dmax.p,
                                  reinterpret_cast<int*>(c->d_ctr.p), FOCK_COUNTER_WORDS, c->st));
    } else {
        HIP_TRY(launch_fock_prep(N, dP, c->d_absD.p, c->d_G.p, c->d_sh_bf0.p, c->d_sh_nbf.p, (int)c->shells.size(),
                                 c->d_Dsh.p, reinterpret_cast<int*>(c->d_ctr.p), FOCK_COUNTER_WORDS, c->st));
    }
    ClassArgs A = base_args(c);
    A.absD = c->d_absD.p;
    A.sqS = c->d_sqS.p;
    A.tol = tol;
    A.D = dP;
    A.G = c->d_G.p;
    FockScratch W;
    W.counters(c->d_ctr.p);
    W.profile_events = true;
    W.Dsh = c->d_Dsh.p;
    if (blocks) {
        UnitLive U;
        for (int qc = 0; qc <= NQCLASS; ++qc) U.off[qc] = c->unit_off[qc];
        U.bound = c->d_ubound.p;
        U.mol_dmax = c->d_mol_dmax.p;
        U.tol = tol;
        U.live = c->d_live.p;
        U.nlive = c->d_ctr.p->nlive;
        HIP_TRY(launch_unit_live(U, c->st));
        W.live = c->d_live.p;
    }
    W.surv = c->d_surv.p;
    W.surv_cap = (int64_t)c->d_surv.n;   // reserved by the caller
    W.allow_measure = false;
    int rc = run_fock_classes(c, A, tol, W);
    if (rc) return rc;
    if (blocks)
        HIP_TRY(launch_block_symmetrize(c->nmol, c->d_mol_blocks.p, N, c->d_G.p, Gout, c->st));
    else
        HIP_TRY(launch_symmetrize(N, c->d_G.p, Gout, c->st));
    return MMD_OK;
}

__global__ void batch_axpy_kernel(size_t n, const double* __restrict__ a, const double* __restrict__ b,
                                  double* __restrict__ out)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = a[i] + b[i];
}
}  // namespace

int mmd_batch_rhf(mmd_ctx* ctx, const int32_t* nocc, const double* enuc, const double* P0, double conver,
                  double acc2e, int maxiter, int diis, int use_graph, double* energy, int32_t* iterations,
                  int32_t* converged, double* P_out, double* mo_out)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    mmd_ctx* c = ctx;
    if (c->nbf == 0) return fail(MMD_ERR_STATE, "no basis set");
    if (!c->shells_ok) return fail(MMD_ERR_UNSUPPORTED, "%s", c->shells_err.c_str());
    if (!nocc || !enuc || !energy || !iterations || !converged || maxiter < 1)
        return fail(MMD_ERR_ARG, "invalid batch arguments");
    const int M = c->nmol, N = c->nbf;
    const size_t nn = (size_t)N * N;
    std::vector<BatchMol> mols(M);
    size_t wtot = 0, dtot = 0, ptot = 0;
    for (int m = 0; m < M; ++m) {
        const int n = c->mol_n[m];
        if (n > BATCH_MAX_NBF)
            return fail(MMD_ERR_UNSUPPORTED, "molecule %d has %d basis functions; the batch takes up to %d", m, n,
                        BATCH_MAX_NBF);
        if (nocc[m] < 1 || nocc[m] > n) return fail(MMD_ERR_ARG, "molecule %d: invalid occupation", m);
        BatchMol& b = mols[m];
        b.f0 = c->mol_f0[m];
        b.n = n;
        b.nocc = nocc[m];
        b.pad = 0;
        b.wo = wtot;
        b.d8 = dtot;
        b.po = ptot;
        b.enuc = enuc[m];
        wtot += 3 * (size_t)n * n;
        dtot += 16 * (size_t)n * n;
        ptot += (size_t)n * n;
    }
    hipStream_t st = c->st;
    // one-electron integrals of every molecule's own block; H = T + V
    HIP_TRY(c->d_onee.reserve(3 * nn));
    double* S = c->d_onee.p;
    {
        const double origin[3] = {0.0, 0.0, 0.0};
        if ((rc = one_electron_shells(c, origin, S, S + nn, S + 2 * nn, nullptr, nullptr))) return rc;
    }
    for (DevBuf<double>* b : {&c->b_H, &c->b_X, &c->b_U, &c->b_F, &c->b_P, &c->b_Pold, &c->b_dP, &c->b_G})
        HIP_TRY(b->reserve(nn));
    HIP_TRY(c->b_diis.reserve(std::max<size_t>(1, dtot)));
    HIP_TRY(c->b_mo.reserve(N));
    HIP_TRY(c->b_state.reserve(M));
    HIP_TRY(c->b_flag.reserve(M));
    HIP_TRY(c->b_count.reserve(1));
    hipLaunchKernelGGL(batch_axpy_kernel, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, st, nn, S + nn, S + 2 * nn,
                       c->b_H.p);
    HIP_TRY(hipGetLastError());
    // Schwarz diagonal, pair tables and work units of the whole batch
    HIP_TRY(c->d_schwarz.reserve(nn));
    if ((rc = schwarz_diagonal(c, c->d_schwarz.p))) return rc;
    HIP_TRY(c->b_mol.reserve(M));
    HIP_TRY(hipMemcpyAsync(c->b_mol.p, mols.data(), sizeof(BatchMol) * M, hipMemcpyHostToDevice, st));
    BatchArgs B;
    B.nmol = M;
    B.N = N;
    B.maxn = c->rw;
    B.lds_bytes = c->lds_per_block;
    B.mol = c->b_mol.p;
    HIP_TRY(c->b_work.reserve(std::max<size_t>(1, wtot)));   // 3 n^2 per molecule: staging for packed blocks
    if ((rc = finish_schwarz(c))) return rc;
    // buffers of the Fock build, reserved before any capture
    {
        int64_t wave = 0;
        for (int qc = 0; qc < NQCLASS; ++qc) {
            int la, lb, lc, ld;
            qclass_decode(qc, &la, &lb, &lc, &ld);
            if (c->qc_total[qc] && fock_class_is_wave(la, lb, lc, ld)) wave += 2 * c->qc_total[qc];
        }
        // survivor lists of the wavefront classes; row-kernel fallbacks need
        // more and are refused by the capacity check
        HIP_TRY(c->d_surv.reserve((size_t)std::max<int64_t>(wave, 1)));
    }
    // state: core guess F = H, P = P_old = 0; or the given densities
    std::vector<BatchState> st0(M);
    for (auto& x : st0) {
        memset(&x, 0, sizeof(x));
        x.energy = 0.0;
        x.prms = 1e20;
    }
    HIP_TRY(hipMemcpyAsync(c->b_state.p, st0.data(), sizeof(BatchState) * M, hipMemcpyHostToDevice, st));
    HIP_TRY(launch_fill_int(M, c->b_flag.p, 0, st));
    HIP_TRY(hipMemcpyAsync(c->b_F.p, c->b_H.p, sizeof(double) * nn, hipMemcpyDeviceToDevice, st));
    HIP_TRY(launch_fill(nn, c->b_P.p, 0.0, st));
    B.state = c->b_state.p;
    B.S = S;
    B.H = c->b_H.p;
    B.X = c->b_X.p;
    B.U = c->b_U.p;
    B.F = c->b_F.p;
    B.P = c->b_P.p;
    B.Pold = c->b_Pold.p;
    B.dP = c->b_dP.p;
    B.G = c->b_G.p;
    B.work = c->b_work.p;
    B.diis = c->b_diis.p;
    B.mo = c->b_mo.p;
    B.flag = c->b_flag.p;
    HIP_TRY(launch_batch_overlap(B, st));
    if (P0) {
        // an initial density (SAD, learned): F = H + G(P0), P_old = P0
        // (packed blocks through the work area, which the steps use later)
        HIP_TRY(hipMemcpyAsync(c->b_work.p, P0, sizeof(double) * ptot, hipMemcpyHostToDevice, st));
        HIP_TRY(launch_batch_unpack(B, c->b_work.p, c->b_P.p, st));
        HIP_TRY(hipStreamSynchronize(st));
        if ((rc = enqueue_fock_sym(c, c->b_P.p, acc2e, c->b_G.p))) return rc;
        hipLaunchKernelGGL(batch_axpy_kernel, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, st, nn, c->b_H.p,
                           c->b_G.p, c->b_F.p);
        HIP_TRY(hipGetLastError());
    }
    HIP_TRY(hipMemcpyAsync(c->b_Pold.p, c->b_P.p, sizeof(double) * nn, hipMemcpyDeviceToDevice, st));
    HIP_TRY(launch_batch_step(B, 0, diis, conver, st));
    {
        std::vector<int> fl(M);
        HIP_TRY(hipMemcpyAsync(fl.data(), c->b_flag.p, sizeof(int) * M, hipMemcpyDeviceToHost, st));
        HIP_TRY(hipStreamSynchronize(st));
        for (int m = 0; m < M; ++m)
            if (fl[m] == -1) return fail(MMD_ERR_ARG, "molecule %d: overlap matrix not positive definite", m);
    }
    // iterations 1 .. maxiter-1: Fock build of the whole batch from dP, then
    // the per-molecule step; replayed from a graph when use_graph
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    auto iteration = [&]() -> int {
        int r = enqueue_fock_sym(c, c->b_dP.p, acc2e, c->b_G.p);
        if (r) return r;
        HIP_TRY(launch_batch_step(B, 1, diis, conver, st));
        return MMD_OK;
    };
    // profiling: per-class events and counters read after every build, so
    // the iterations are launched one by one
    const bool profiled = c->profiling != 0;
    if (use_graph && !profiled) {
        std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
        if (hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed) == hipSuccess) {
            const int r = iteration();
            hipGraph_t g = nullptr;
            const hipError_t e = hipStreamEndCapture(st, &g);
            if (r == MMD_OK && e == hipSuccess && g &&
                hipGraphInstantiate(&exec, g, nullptr, nullptr, 0) == hipSuccess) {
                graph = g;
            } else {
                if (g) (void)hipGraphDestroy(g);
                exec = nullptr;
                (void)hipGetLastError();
                if (r) return r;
            }
        }
    }
    int left = M;
    for (int it = 1; it < maxiter && left > 0; ++it) {
        if (exec) {
            HIP_TRY(hipGraphLaunch(exec, st));
        } else if ((rc = iteration())) {
            return rc;
        }
        if (profiled && (rc = collect_profile(c))) return rc;
        if (it % 4 == 0 || it == maxiter - 1) {
            HIP_TRY(launch_batch_count(B, c->b_count.p, st));
            HIP_TRY(hipMemcpyAsync(&left, c->b_count.p, sizeof(int), hipMemcpyDeviceToHost, st));
            HIP_TRY(hipStreamSynchronize(st));
        }
    }
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    std::vector<BatchState> out(M);
    std::vector<int> fl(M);
    HIP_TRY(hipMemcpyAsync(out.data(), c->b_state.p, sizeof(BatchState) * M, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipMemcpyAsync(fl.data(), c->b_flag.p, sizeof(int) * M, hipMemcpyDeviceToHost, st));
    if (mo_out) HIP_TRY(hipMemcpyAsync(mo_out, c->b_mo.p, sizeof(double) * N, hipMemcpyDeviceToHost, st));
    if (P_out) {
        HIP_TRY(launch_batch_pack(B, c->b_P.p, c->b_work.p, st));
        HIP_TRY(hipMemcpyAsync(P_out, c->b_work.p, sizeof(double) * ptot, hipMemcpyDeviceToHost, st));
    }
    HIP_TRY(hipStreamSynchronize(st));
    for (int m = 0; m < M; ++m) {
        if (fl[m] == -2) return fail(MMD_ERR_STATE, "molecule %d: singular DIIS matrix", m);
        energy[m] = out[m].energy;
        iterations[m] = out[m].iterations;
        converged[m] = out[m].converged;
    }
    return MMD_OK;
}

int mmd_scf_begin(mmd_ctx* ctx, int nocc, const double* H, const double* S, const double* X, const double* F,
                  const double* P)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    const int N = ctx->nbf;
    if (N == 0) return fail(MMD_ERR_STATE, "no basis set");
    if (nocc < 1 || nocc > N || !H || !S || !X || !F || !P) return fail(MMD_ERR_ARG, "invalid SCF arguments");
    if (!ctx->blas) {
        std::lock_guard<std::recursive_mutex> lk(device_alloc_mutex());
        if (rocblas_create_handle(&ctx->blas) != rocblas_status_success)
            return fail(MMD_ERR_DEVICE, "rocblas_create_handle failed");
    }
    if (rocblas_set_stream(ctx->blas, ctx->st) != rocblas_status_success)
        return fail(MMD_ERR_DEVICE, "rocblas_set_stream failed");
    const size_t nn = (size_t)N * N;
    for (DevBuf<double>* b : {&ctx->s_H, &ctx->s_S, &ctx->s_X, &ctx->s_F, &ctx->s_P, &ctx->s_Pold, &ctx->s_G,
                              &ctx->s_dP, &ctx->s_T1, &ctx->s_T2, &ctx->s_C})
        HIP_TRY(b->reserve(nn));
    HIP_TRY(ctx->s_Fset.reserve(8 * nn));
    HIP_TRY(ctx->s_Eset.reserve(8 * nn));
    HIP_TRY(ctx->s_stats.reserve(2));
    HIP_TRY(ctx->s_dots.reserve(8));
    const size_t by = sizeof(double) * nn;
    HIP_TRY(hipMemcpyAsync(ctx->s_H.p, H, by, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(ctx->s_S.p, S, by, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(ctx->s_X.p, X, by, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(ctx->s_F.p, F, by, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(ctx->s_P.p, P, by, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(ctx->s_Pold.p, P, by, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(launch_fill(nn, ctx->s_G.p, 0.0, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    ctx->scf_n = N;
    ctx->scf_nocc = nocc;
    ctx->s_order.clear();
    ctx->s_B.assign(64, 0.0);
    return MMD_OK;
}

int mmd_scf_step(mmd_ctx* ctx, double tol, int build, int diis, double* FO)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if ((rc = scf_check(ctx))) return rc;
    if (!FO) return fail(MMD_ERR_ARG, "null pointer");
    const int N = ctx->nbf;
    const size_t nn = (size_t)N * N;
    hipStream_t st = ctx->st;
    const double* Fuse = ctx->s_F.p;
    if (build) {
        // F <- F + G(P - P_old); P_old <- P   (mmd/scf.py:84-94)
        HIP_TRY(launch_scf_axpby(nn, 1.0, ctx->s_P.p, -1.0, ctx->s_Pold.p, ctx->s_dP.p, st));
        rc = mmd_fock_delta(ctx, ctx->s_dP.p, nullptr, tol, 0, ctx->s_G.p, nullptr, 1, nullptr);
        if (rc) return rc;
        HIP_TRY(launch_scf_axpby(nn, 1.0, ctx->s_F.p, 1.0, ctx->s_G.p, ctx->s_F.p, st));
        HIP_TRY(hipMemcpyAsync(ctx->s_Pold.p, ctx->s_P.p, sizeof(double) * nn, hipMemcpyDeviceToDevice, st));
        if (diis) {
            // error X (FPS - SPF) X of the new F, into the window (mmd/scf.py:146-180)
            int slot;
            std::vector<int>& ord = ctx->s_order;
            std::vector<double>& B = ctx->s_B;
            if ((int)ord.size() == 8) {
                slot = ord.front();
                ord.erase(ord.begin());
                for (int i = 0; i < 7; ++i)
                    for (int j = 0; j < 7; ++j) B[i * 8 + j] = B[(i + 1) * 8 + (j + 1)];
            } else {
                slot = (int)ord.size();
            }
            double* Es = ctx->s_Eset.p + (size_t)slot * nn;
            double* Fs = ctx->s_Fset.p + (size_t)slot * nn;
            if ((rc = gemm_rm(ctx, false, false, N, N, N, ctx->s_P.p, N, ctx->s_S.p, N, ctx->s_T1.p, N))) return rc;
            if ((rc = gemm_rm(ctx, false, false, N, N, N, ctx->s_F.p, N, ctx->s_T1.p, N, ctx->s_T2.p, N))) return rc;
            HIP_TRY(launch_scf_antisym(N, ctx->s_T2.p, ctx->s_T1.p, st));
            if ((rc = gemm_rm(ctx, false, false, N, N, N, ctx->s_X.p, N, ctx->s_T1.p, N, ctx->s_T2.p, N))) return rc;
            if ((rc = gemm_rm(ctx, false, false, N, N, N, ctx->s_T2.p, N, ctx->s_X.p, N, Es, N))) return rc;
            HIP_TRY(hipMemcpyAsync(Fs, ctx->s_F.p, sizeof(double) * nn, hipMemcpyDeviceToDevice, st));
            ord.push_back(slot);
            const int n = (int)ord.size();
            const double* E[8];
            const double* Fk[8];
            for (int k = 0; k < n; ++k) {
                E[k] = ctx->s_Eset.p + (size_t)ord[k] * nn;
                Fk[k] = ctx->s_Fset.p + (size_t)ord[k] * nn;
            }
            double dots[8];
            HIP_TRY(launch_scf_dots(n, nn, E, Es, ctx->s_dots.p, st));
            HIP_TRY(hipMemcpyAsync(dots, ctx->s_dots.p, sizeof(double) * n, hipMemcpyDeviceToHost, st));
            HIP_TRY(hipStreamSynchronize(st));
            for (int k = 0; k < n; ++k) B[(n - 1) * 8 + k] = B[k * 8 + (n - 1)] = dots[k];
            // [B -1; -1 0] w = [0 .. 0 -1]
            const int m = n + 1;
            std::vector<double> A((size_t)m * m, 0.0), w(m, 0.0);
            for (int i = 0; i < n; ++i)
                for (int j = 0; j < n; ++j) A[i * m + j] = B[i * 8 + j];
            for (int i = 0; i < n; ++i) A[i * m + n] = A[n * m + i] = -1.0;
            w[n] = -1.0;
            if (!solve_small(m, A, w)) return fail(MMD_ERR_STATE, "singular DIIS matrix");
            double sw = 0.0;
            for (int k = 0; k < n; ++k) sw += w[k];
            if (!(fabs(sw - 1.0) <= 1e-8 + 1e-5)) return fail(MMD_ERR_STATE, "DIIS weights do not sum to one");
            HIP_TRY(launch_scf_combine(nn, n, Fk, w.data(), ctx->s_C.p, st));
            Fuse = ctx->s_C.p;
        }
    }
    // FO = X^T F X
    if ((rc = gemm_rm(ctx, true, false, N, N, N, ctx->s_X.p, N, Fuse, N, ctx->s_T1.p, N))) return rc;
    if ((rc = gemm_rm(ctx, false, false, N, N, N, ctx->s_T1.p, N, ctx->s_X.p, N, ctx->s_T2.p, N))) return rc;
    HIP_TRY(hipMemcpyAsync(FO, ctx->s_T2.p, sizeof(double) * nn, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    return MMD_OK;
}

int mmd_scf_density(mmd_ctx* ctx, const double* CO, double* stats)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if ((rc = scf_check(ctx))) return rc;
    if (!CO || !stats) return fail(MMD_ERR_ARG, "null pointer");
    const int N = ctx->nbf;
    const size_t nn = (size_t)N * N;
    hipStream_t st = ctx->st;
    // C = X C'; P = C_occ C_occ^T; E_el = sum (H + F)_pq P_qp; ||P - P_old||^2
    HIP_TRY(hipMemcpyAsync(ctx->s_T1.p, CO, sizeof(double) * nn, hipMemcpyHostToDevice, st));
    if ((rc = gemm_rm(ctx, false, false, N, N, N, ctx->s_X.p, N, ctx->s_T1.p, N, ctx->s_T2.p, N))) return rc;
    if ((rc = gemm_rm(ctx, false, true, N, N, ctx->scf_nocc, ctx->s_T2.p, N, ctx->s_T2.p, N, ctx->s_P.p, N)))
        return rc;
    HIP_TRY(launch_scf_energy(N, ctx->s_H.p, ctx->s_F.p, ctx->s_P.p, ctx->s_Pold.p, ctx->s_stats.p, st));
    double h[2];
    HIP_TRY(hipMemcpyAsync(h, ctx->s_stats.p, sizeof(h), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    stats[0] = h[0];
    stats[1] = sqrt(h[1]);
    return MMD_OK;
}

int mmd_scf_get(mmd_ctx* ctx, double* F, double* P, double* P_old, double* G)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if ((rc = scf_check(ctx))) return rc;
    const size_t by = sizeof(double) * (size_t)ctx->nbf * ctx->nbf;
    if (F) HIP_TRY(hipMemcpyAsync(F, ctx->s_F.p, by, hipMemcpyDeviceToHost, ctx->st));
    if (P) HIP_TRY(hipMemcpyAsync(P, ctx->s_P.p, by, hipMemcpyDeviceToHost, ctx->st));
    if (P_old) HIP_TRY(hipMemcpyAsync(P_old, ctx->s_Pold.p, by, hipMemcpyDeviceToHost, ctx->st));
    if (G) HIP_TRY(hipMemcpyAsync(G, ctx->s_G.p, by, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    return MMD_OK;
}

int mmd_ao2mo(mmd_ctx* ctx, const double* T, int t_on_device, const double* C, double* out, int out_on_device,
              double* gemm_ms)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (ctx->nbf == 0) return fail(MMD_ERR_STATE, "no basis set");
    if (!T || !C || !out) return fail(MMD_ERR_ARG, "null pointer");
    const int N = ctx->nbf;
    const size_t nn = (size_t)N * N, n3 = nn * N, n4 = nn * nn;
    if (n3 > (size_t)INT32_MAX) return fail(MMD_ERR_UNSUPPORTED, "basis too large for the transform");
    Tensor4 a, b;
    HostStage stage;
    DevBuf<double>& dC = ctx->jk_mats;
    HIP_TRY(a.reserve(n4));
    HIP_TRY(b.reserve(n4));
    HIP_TRY(dC.reserve(nn));
    HIP_TRY(hipMemcpyAsync(dC.p, C, sizeof(double) * nn, hipMemcpyHostToDevice, ctx->st));
    if (t_on_device)
        HIP_TRY(hipMemcpyAsync(a.p, T, sizeof(double) * n4, hipMemcpyDeviceToDevice, ctx->st));
    else
        HIP_TRY(stage.to_device(a.p, T, sizeof(double) * n4, ctx->st));
    // Four quarter transforms.  Each contracts the last index of X (M x N,
    // M = N^3) with C and writes it first: Y[S][pqr] = sum_s C[s][S] X[pqr][s],
    // i.e. Y = C^T X^T; after four passes the index order is (P,Q,R,S) again.
    double* x = a.p;
    double* y = b.p;
    HIP_TRY(hipEventRecord(ctx->ev0, ctx->st));
    for (int pass = 0; pass < 4; ++pass) {
        HIP_TRY(launch_gemm_f64(true, true, N, (int)n3, N, 1.0, dC.p, N, x, N, 0.0, y, (int)n3, ctx->st));
        std::swap(x, y);
    }
    HIP_TRY(hipEventRecord(ctx->ev1, ctx->st));
    if (out_on_device)
        HIP_TRY(hipMemcpyAsync(out, x, sizeof(double) * n4, hipMemcpyDeviceToDevice, ctx->st));
    else
        HIP_TRY(stage.to_host(out, x, sizeof(double) * n4, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    a.done();
    b.done();
    stage.done();
    if (gemm_ms) {
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        *gemm_ms = ms;
    }
    return MMD_OK;
}

int mmd_overlap_powers(mmd_ctx* ctx, const double* S, double* X, double* U, int* iterations)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (ctx->nbf == 0) return fail(MMD_ERR_STATE, "no basis set");
    if (!X && !U) return fail(MMD_ERR_ARG, "null pointer");
    const int N = ctx->nbf;
    const size_t nn = (size_t)N * N;
    if (!S && ctx->d_onee.n < nn) return fail(MMD_ERR_STATE, "no overlap matrix: call mmd_one_electron or pass S");
    HIP_TRY(ctx->d_ns.reserve(8 * nn + 2));
    double* dS = ctx->d_ns.p;
    double* dX = dS + nn;
    double* dU = dX + nn;
    if (S)
        HIP_TRY(hipMemcpyAsync(dS, S, sizeof(double) * nn, hipMemcpyHostToDevice, ctx->st));
    else   // the overlap of the last mmd_one_electron, still on the device
        HIP_TRY(hipMemcpyAsync(dS, ctx->d_onee.p, sizeof(double) * nn, hipMemcpyDeviceToDevice, ctx->st));
    const int it = overlap_powers_device(N, dS, dX, dU, dU + nn, 100, ctx->st);
    if (it < 0) return fail(MMD_ERR_DEVICE, "overlap powers: kernel launch failed");
    if (it == 0)
        return fail(MMD_ERR_ARG, "overlap matrix is not positive definite (Newton-Schulz did not converge)");
    if (X) HIP_TRY(hipMemcpyAsync(X, dX, sizeof(double) * nn, hipMemcpyDeviceToHost, ctx->st));
    if (U) HIP_TRY(hipMemcpyAsync(U, dU, sizeof(double) * nn, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    if (iterations) *iterations = it;
    return MMD_OK;
}

int mmd_dgemm(mmd_ctx* ctx, int transA, int transB, int M, int N, int K, double alpha, const double* A, int lda,
              const double* B, int ldb, double beta, double* C, int ldc, int on_device)
{
    int rc = check_ctx(ctx);
    if (rc) return rc;
    if (M < 0 || N < 0 || K < 0) return fail(MMD_ERR_ARG, "negative dimension");
    if (!A || !B || !C) return fail(MMD_ERR_ARG, "null pointer");
    const int rA = transA ? K : M, cA = transA ? M : K;
    const int rB = transB ? N : K, cB = transB ? K : N;
    if (lda < std::max(1, cA) || ldb < std::max(1, cB) || ldc < std::max(1, N))
        return fail(MMD_ERR_ARG, "leading dimension too small");
    if (on_device) {
        HIP_TRY(launch_gemm_f64(transA, transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, ctx->st));
        HIP_TRY(hipStreamSynchronize(ctx->st));
        return MMD_OK;
    }
    const size_t nA = (size_t)rA * lda, nB = (size_t)rB * ldb, nC = (size_t)M * ldc;
    DevBuf<double> a, b, c;
    HIP_TRY(a.reserve(nA));
    HIP_TRY(b.reserve(nB));
    HIP_TRY(c.reserve(nC));
    HIP_TRY(hipMemcpyAsync(a.p, A, sizeof(double) * nA, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(b.p, B, sizeof(double) * nB, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(hipMemcpyAsync(c.p, C, sizeof(double) * nC, hipMemcpyHostToDevice, ctx->st));
    HIP_TRY(launch_gemm_f64(transA, transB, M, N, K, alpha, a.p, lda, b.p, ldb, beta, c.p, ldc, ctx->st));
    HIP_TRY(hipMemcpyAsync(C, c.p, sizeof(double) * nC, hipMemcpyDeviceToHost, ctx->st));
    HIP_TRY(hipStreamSynchronize(ctx->st));
    return MMD_OK;
}

int mmd_last_fock_ms(mmd_ctx* ctx, double* ms)
{
    if (!ctx || !ms) return fail(MMD_ERR_ARG, "null pointer");
    *ms = ctx->last_fock_ms;
    return MMD_OK;
}

}  // extern "C"
