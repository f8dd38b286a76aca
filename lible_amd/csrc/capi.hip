// The C-ABI of lbx (include/lbx.h): context set-up, Schwarz screening, task tables and the
// drivers that launch the quartet kernels class pair by class pair.
#include "grad.hpp"
#include "lbx_internal.hpp"
#include "quartet.hpp"
#include "registry.hpp"
#include "tasks.hpp"
#include "variant_cost.hpp"

#include <algorithm>
#include <cmath>
#include <limits>
#include <map>
#include <memory>
#include <numeric>
#include <string>
#include <tuple>
#include <unordered_map>

// Staging area of the allocation-free block entry (lbx_eri4_batch_static): one call's task list,
// four ints per entry, at most kStaticEntries entries (16 MiB).  Each device holds its own copy
// for the life of the process.  Host code never passes this name to a kernel or a copy: it uses
// the address hipGetSymbolAddress returned for the device (scratchAddress below).
constexpr long long kStaticEntries = 1LL << 20;
static __device__ __align__(256) int scratch[4 * kStaticEntries];

namespace lbx
{
    namespace
    {
        thread_local std::string g_err;

        // scratch device buffer owned by one call
        struct DevBuf
        {
            double *p = nullptr;
            explicit DevBuf(size_t n) { LBX_HIP(hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(double))); }
            ~DevBuf()
            {
                if (p)
                    (void)hipFree(p);
            }
            DevBuf(const DevBuf &) = delete;
            DevBuf &operator=(const DevBuf &) = delete;
        };

        // The extra streams of a context (default priority) and the events that tie them to its
        // stream; made on first use.
        struct SideStreams
        {
            static constexpr int kCount = 3;
            hipStream_t s[kCount] = {};
            hipEvent_t fork = nullptr, joined[kCount] = {};

            void ensure()
            {
                for (int i = 0; i < kCount; i++)
                {
                    if (!s[i])
                        LBX_HIP(hipStreamCreateWithFlags(&s[i], hipStreamNonBlocking));
                    if (!joined[i])
                        LBX_HIP(hipEventCreateWithFlags(&joined[i], hipEventDisableTiming));
                }
                if (!fork)
                    LBX_HIP(hipEventCreateWithFlags(&fork, hipEventDisableTiming));
            }
            ~SideStreams()
            {
                for (int i = 0; i < kCount; i++)
                {
                    if (s[i])
                        (void)hipStreamDestroy(s[i]);
                    if (joined[i])
                        (void)hipEventDestroy(joined[i]);
                }
                if (fork)
                    (void)hipEventDestroy(fork);
            }
        };

        template <class F>
        int guarded(F &&f)
        {
            try
            {
                f();
                return LBX_OK;
            }
            catch (const Error &e)
            {
                g_err = e.what();
                return e.code;
            }
            catch (const std::exception &e)
            {
                g_err = e.what();
                return LBX_ERR_INVALID;
            }
        }

        __global__ void fillKernel(double *p, long long n, double v)
        {
            for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
                 i += static_cast<long long>(gridDim.x) * blockDim.x)
                p[i] = v;
        }

        // M <- S + S^T for an n x n row-major matrix, S = M + its further parts
        __global__ void symmetrizeKernel(double *M, int n, const double *parts, int nparts)
        {
            const long long tot = static_cast<long long>(n) * n;
            for (long long e = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; e < tot;
                 e += static_cast<long long>(gridDim.x) * blockDim.x)
            {
                const int i = static_cast<int>(e / n), j = static_cast<int>(e % n);
                if (j < i)
                    continue;
                const long long t = static_cast<long long>(j) * n + i;
                double v = M[e] + M[t];
                for (int k = 0; k < nparts; k++)
                    v += parts[k * tot + e] + parts[k * tot + t];
                M[e] = v;
                M[t] = v;
            }
        }

        // out[i] = sum over the copies of in[copy * n + i]
        __global__ void sumCopiesKernel(const double *in, double *out, long long n, int copies)
        {
            const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
            if (i >= n)
                return;
            double s = 0.0;
            for (int k = 0; k < copies; k++)
                s += in[k * n + i];
            out[i] = s;
        }

        void fill(double *p, long long n, double v, hipStream_t s)
        {
            if (n <= 0)
                return;
            long long b = (n + 255) / 256;
            hipLaunchKernelGGL(fillKernel, dim3(static_cast<int>(std::min(b, 65536LL))), dim3(256), 0, s,
                               p, n, v);
            LBX_HIP(hipGetLastError());
        }

        // Device address of the scratch array on device dev, looked up once per device with that
        // device current (context set-up) and kept for every later context on it
        int *scratchAddress(int dev)
        {
            static std::mutex m;
            static std::map<int, int *> addr;
            std::lock_guard<std::mutex> lk(m);
            auto it = addr.find(dev);
            if (it != addr.end())
                return it->second;
            void *p = nullptr;
            LBX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
            if (!p)
                throw Error(LBX_ERR_HIP, "hipGetSymbolAddress(scratch) returned a null address");
            addr[dev] = static_cast<int *>(p);
            return static_cast<int *>(p);
        }

        // Boys table, one copy per device for the life of the process
        const double *boysTableDevice()
        {
            static std::mutex m;
            static std::map<int, double *> tabs;
            int dev = 0;
            LBX_HIP(hipGetDevice(&dev));
            std::lock_guard<std::mutex> lk(m);
            auto it = tabs.find(dev);
            if (it != tabs.end())
                return it->second;
            auto h = boysTable();
            double *d = nullptr;
            LBX_HIP(hipMalloc(&d, h.size() * sizeof(double)));
            LBX_HIP(hipMemcpy(d, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice));
            tabs[dev] = d;
            return d;
        }

        template <int N>
        __global__ void boysKernel(long long cnt, const double *x, double *out, const double *tab)
        {
            for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < cnt;
                 i += static_cast<long long>(gridDim.x) * blockDim.x)
            {
                double F[N + 1];
                boysF<N>(x[i], tab, F);
                for (int k = 0; k <= N; k++)
                    out[i * (N + 1) + k] = F[k];
            }
        }

        template <int N>
        void launchBoys(long long cnt, const double *x, double *out, const double *tab, hipStream_t s)
        {
            long long b = (cnt + 255) / 256;
            hipLaunchKernelGGL((boysKernel<N>), dim3(static_cast<int>(std::min(b, 65536LL))), dim3(256),
                               0, s, cnt, x, out, tab);
        }

        using BoysFn = void (*)(long long, const double *, double *, const double *, hipStream_t);
        template <int... Ns>
        constexpr std::array<BoysFn, sizeof...(Ns)> boysFns(std::integer_sequence<int, Ns...>)
        {
            return {&launchBoys<Ns>...};
        }

        // ------------------------------------------------------------------ task tables
        struct TaskTable
        {
            long long ntasks = 0;
            int nket = 0;
            std::vector<long long> prefix;
            std::vector<int> plo, phi;
            tasks::Cuts cuts;   // the Schwarz cuts behind plo/phi (buildTasks)
            long long *d_prefix = nullptr;
            int *d_plo = nullptr, *d_phi = nullptr;
            double quartets = 0, flops = 0;
            // over the quartets: sum of K_bra K_ket, of K_bra, of K_ket (canonical roles)
            double sum_kk = 0, sum_kbra = 0, sum_kket = 0;
            // lane-block-major enumeration of a 64-wide table (empty unless built)
            int nblk = 0, gshift = 0;
            long long btasks = 0;
            std::vector<long long> bprefix;
            std::vector<int> bq0;
            long long *d_bprefix = nullptr;
            int *d_bq0 = nullptr;
        };

        enum class Pairing
        {
            Unique,     // p >= q when bra and ket are the same class, all p otherwise
            All,        // every (p, q)
            Diagonal    // p == q only
        };

        using tasks::firstBelow;

        constexpr double kNoUpper = std::numeric_limits<double>::infinity();
        // quartets per class pair and variant that the autotuner times
        constexpr long long kTuneSample = 2LL << 20;

        // Lane-side positions [plo, phi) per uniform-side position q, with the Schwarz cut
        // thresh <= Q_p Q_q < thresh_hi on descending-sorted Q (thresh <= 0: no lower cut).
        // `bra` is the lane side and `ket` the uniform side; lane_is_bra says whether that
        // matches the canonical (bra class >= ket class) roles, which the FLOP count follows.
        TaskTable buildTasks(Context &c, const PairClass &bra, const PairClass &ket, Pairing mode,
                             bool same, double thresh, int width, bool lane_is_bra = true,
                             double thresh_hi = kNoUpper)
        {
            TaskTable t;
            t.nket = ket.n_pairs;
            t.plo.resize(t.nket);
            t.phi.resize(t.nket);
            t.prefix.resize(t.nket + 1);
            std::vector<double> qb(bra.n_pairs), kab_prefix(bra.n_pairs + 1, 0.0);
            for (int i = 0; i < bra.n_pairs; i++)
            {
                qb[i] = bra.Q.empty() ? 1.0 : bra.Q[bra.order[i]];
                kab_prefix[i + 1] = kab_prefix[i] + bra.pcnt[bra.order[i]];
            }
            const PairClass &cb = lane_is_bra ? bra : ket, &ck = lane_is_bra ? ket : bra;
            const int la = cb.la, lb = cb.lb, lc = ck.la, ld = ck.lb;
            const double Hab = nHerm(la + lb), Hcd = nHerm(lc + ld);
            const double Sab = nSph(la) * nSph(lb), Scd = nSph(lc) * nSph(ld);
            const double perKK = quartetFlops(la, lb, lc, ld, 1, 1) - 2 * Sab * Hab * Scd - 12 * Sab * Scd;
            if (mode != Pairing::Diagonal)
            {
                std::vector<double> qk(t.nket);
                for (int q = 0; q < t.nket; q++)
                    qk[q] = ket.Q.empty() ? 1.0 : ket.Q[ket.order[q]];
                t.cuts = tasks::cut(qb, qk, mode == Pairing::Unique && same, thresh, thresh_hi);
            }
            long long acc = 0;
            for (int q = 0; q < t.nket; q++)
            {
                int lo, hi;
                if (mode == Pairing::Diagonal)
                {
                    lo = q;
                    hi = q + 1;
                }
                else
                {
                    lo = t.cuts.plo[q];
                    hi = t.cuts.phi[q];
                }
                t.plo[q] = lo;
                t.phi[q] = hi;
                t.prefix[q] = acc;
                const long long cnt = hi - lo;
                acc += (cnt + width - 1) / width;
                if (cnt > 0)
                {
                    const double kq = ket.pcnt[ket.order[q]];
                    const double skl = kab_prefix[hi] - kab_prefix[lo];
                    t.quartets += cnt;
                    t.sum_kk += kq * skl;
                    t.sum_kbra += lane_is_bra ? skl : kq * cnt;
                    t.sum_kket += lane_is_bra ? kq * cnt : skl;
                    if (lane_is_bra)
                        t.flops += perKK * kq * skl + 2 * Sab * Hab * Scd * skl + 12 * Sab * Scd * cnt;
                    else
                        t.flops += perKK * kq * skl + 2 * Sab * Hab * Scd * kq * cnt + 12 * Sab * Scd * cnt;
                }
            }
            t.prefix[t.nket] = acc;
            t.ntasks = acc;
            t.d_prefix = c.stage(t.prefix);
            t.d_plo = c.stage(t.plo);
            t.d_phi = c.stage(t.phi);
            return t;
        }

        // Lane-block-major enumeration of a 64-wide table.  Lane block b = positions 64b .. 64b+63,
        // group g = blocks g G .. g G + G - 1 (G = 2^gshift).  Group g takes the uniform positions
        // q = bq0[g] .. bq0[g] + n_g - 1, the smallest range holding every q whose [plo, phi)
        // meets the group, each q with the group's G blocks in turn: G n_g tasks (a task whose
        // block misses q's range has every lane idle and returns at once).  Only groups with
        // g % stride == 0 get tasks (the autotuner's samples); returns the quartets they hold.
        // With a shell-ordered lane side (perm: lane position -> Schwarz-order position) a group
        // holds a subset of the Schwarz-order positions [lowest, highest]: its q range is then
        // conservative (the kernel tests each lane) and its quartets are counted exactly.
        double buildBlockMajor(Context &c, TaskTable &t, int nlane, int stride, int gshift,
                               const std::vector<int> &perm, const std::vector<int> &bqlo,
                               const std::vector<int> &bqhi)
        {
            if (t.cuts.plo.size() != static_cast<size_t>(t.nket))
                throw Error(LBX_ERR_STATE, "lane-block-major table without Schwarz cuts");
            tasks::BlockMajor b = tasks::blockMajor(t.cuts, nlane, stride, gshift, perm);
            try
            {
                tasks::checkBlockMajor(b, t.nket, nlane, gshift, perm, bqlo, bqhi);
            }
            catch (const std::runtime_error &e)
            {
                throw Error(LBX_ERR_STATE, e.what());
            }
            t.gshift = gshift;
            t.bprefix = std::move(b.bprefix);
            t.bq0 = std::move(b.bq0);
            t.btasks = b.ntasks;
            t.d_bprefix = c.stage(t.bprefix);
            t.d_bq0 = c.stage(t.bq0);
            t.nblk = b.nblk;   // the table is there (staging may run out of memory)
            return b.quartets;
        }

        // Tasks of the batched RI sums: for every uniform-side position q the lane-side pairs of
        // q's molecule (each molecule's positions are contiguous), with `same` only lane
        // positions p >= q, and with bounds (both sides sorted by Q within each molecule) only
        // those with lo <= Q_p Q_q < hi.  No screening below: every triplet of the tensors.
        TaskTable buildTasksMol(Context &c, const PairClass &lane, const PairClass &unif, bool same,
                                int width, double lo_bound = 0.0, double hi_bound = kNoUpper,
                                bool staged = true)
        {
            const bool bounded = lo_bound > 0.0 || hi_bound < kNoUpper;
            auto qOf = [](const PairClass &pc, int pos) { return pc.Q.empty() ? 1.0 : pc.Q[pc.order[pos]]; };
            // first position in [a, b) whose bound with qk falls below thr (Q descending there)
            auto firstBelowIn = [&](int a, int b, double qk, double thr) {
                while (a < b)
                {
                    const int m = (a + b) / 2;
                    if (qOf(lane, m) * qk >= thr)
                        a = m + 1;
                    else
                        b = m;
                }
                return a;
            };
            TaskTable t;
            t.nket = unif.n_pairs;
            t.plo.resize(t.nket);
            t.phi.resize(t.nket);
            t.prefix.resize(t.nket + 1);
            std::vector<int> lo(c.nmol, 0), hi(c.nmol, 0);
            std::vector<double> kl_prefix(lane.n_pairs + 1, 0.0);
            for (int p = lane.n_pairs; p-- > 0;)
                lo[lane.mol[lane.order[p]]] = p;
            for (int p = 0; p < lane.n_pairs; p++)
            {
                hi[lane.mol[lane.order[p]]] = p + 1;
                kl_prefix[p + 1] = kl_prefix[p] + lane.pcnt[lane.order[p]];
            }
            const int la = lane.la, lb = lane.lb, lc = unif.la, ld = unif.lb;
            const double Hab = nHerm(la + lb), Sab = nSph(la) * nSph(lb), Scd = nSph(lc) * nSph(ld);
            const double perKK = quartetFlops(la, lb, lc, ld, 1, 1) - 2 * Sab * Hab * Scd - 12 * Sab * Scd;
            long long acc = 0;
            for (int q = 0; q < t.nket; q++)
            {
                const int m = unif.mol[unif.order[q]];
                int a = hi[m] > 0 ? lo[m] : 0, b = hi[m];
                if (bounded && b > a)
                {
                    const double qk = qOf(unif, q);
                    const int a0 = a, b0 = b;
                    if (hi_bound < kNoUpper)
                        a = firstBelowIn(a0, b0, qk, hi_bound);
                    if (lo_bound > 0.0)
                        b = firstBelowIn(a0, b0, qk, lo_bound);
                }
                if (same)
                    a = std::max(a, q);
                b = std::max(a, b);
                t.plo[q] = a;
                t.phi[q] = b;
                t.prefix[q] = acc;
                const long long cnt = b - a;
                // the one-lane form's tasks are the aligned blocks of 64 positions
                acc += width == 64 && cnt > 0 ? (b - (a & ~63) + 63) / 64 : (cnt + width - 1) / width;
                if (cnt > 0)
                {
                    const double kq = unif.pcnt[unif.order[q]];
                    const double skl = kl_prefix[b] - kl_prefix[a];
                    t.quartets += cnt;
                    t.sum_kk += kq * skl;
                    t.sum_kbra += skl;
                    t.sum_kket += kq * cnt;
                    // transforms, R and Boys as for J/K; the epilogue sums 2 values per element
                    t.flops += perKK * kq * skl + 2 * Sab * Hab * Scd * skl + 2 * Sab * Scd * cnt;
                }
            }
            t.prefix[t.nket] = acc;
            t.ntasks = acc;
            // staged arrays stay with the context, uploaded ones can be freed one by one
            t.d_prefix = staged ? c.stage(t.prefix) : c.upload(t.prefix);
            t.d_plo = staged ? c.stage(t.plo) : c.upload(t.plo);
            t.d_phi = staged ? c.stage(t.phi) : c.upload(t.phi);
            return t;
        }

        void requireSingle(const Context &c, const char *who)
        {
            if (!c.atom_mol.empty())
                throw Error(LBX_ERR_STATE, std::string(who) + ": not available on a batched context "
                                                              "(pairs only exist within each molecule)");
        }

        KArgs baseArgs(Context &c, const PairClass &bra, const PairClass &ket, const TaskTable &t,
                       bool same)
        {
            KArgs a{};
            a.bra = bra.view();
            a.ket = ket.view();
            a.prefix = t.d_prefix;
            a.plo = t.d_plo;
            a.phi = t.d_phi;
            a.nket = t.nket;
            a.ntasks = t.ntasks;
            a.same_class = same ? 1 : 0;
            a.boys = c.d_boys;
            a.nbf = static_cast<long long>(c.nbf);
            a.naux = static_cast<long long>(c.nbf_aux);
            return a;
        }

        int rFlopsHost(int L)
        {
            int r = 0;
            for (int n = 0; n < L; n++)
                for (int m = 1; m <= L - n; m++)
                    r += (m + 1) * (m + 2) / 2;
            return 2 * r;
        }

        // primitive pairs per shell pair of a class, as the time estimates take them
        cost::Side costSide(const PairClass &pc)
        {
            const double kmean = pc.n_pairs ? double(pc.n_ppairs) / pc.n_pairs : 1.0;
            return {pc.la, pc.lb, kmean, pc.klane > 0 ? pc.klane : 0.5 * (kmean + pc.kmax), std::max<double>(pc.kmax, 1.0)};
        }

        // Estimated time (ms) of one form over `quartets` quartets, which a one-lane form takes in
        // `waves` tasks.
        double variantTime(int mode, const PairClass &bra, const PairClass &ket, const KernelSlot &s, bool f32,
                           double quartets, double waves)
        {
            const cost::Side b = costSide(bra), k = costSide(ket);
            if (s.kind == KIND_LANE)
                return cost::laneForm(s.swap ? k : b, s.swap ? b : k, s.nc, f32, waves, mode == MODE_JK || mode == MODE_SUM, mode == MODE_JK);
            return s.kind == KIND_WAVE ? cost::waveForm(b, k, f32, quartets) : cost::blockForm(b, k, f32, quartets);
        }

        // Whether the kernel of a variant is a form of its own: a one-lane number whose form is not built
        // runs the one-wave form, which has a number already.
        bool ownForm(int v, const KernelSlot &s)
        {
            const bool laneVariant = v != VAR_MFMA && v != VAR_MFMA32 && v != VAR_BLOCK && v != VAR_BLOCK32;
            return s.fn && laneVariant == (s.kind == KIND_LANE);
        }

        // The form with the smallest estimate among the FP64 (or FP32) ones, and that estimate; -1
        // when the class pair has none.  wavesBra, wavesKet: tasks of the one-lane forms with the
        // bra (ket) pairs on the lanes.
        int defaultVariant(int mode, const PairClass &bra, const PairClass &ket, bool f32, double quartets,
                           double wavesBra, double wavesKet, double *ms = nullptr)
        {
            int best = -1;
            double tBest = 0.0;
            for (int v = 0; v < N_VARIANTS; v++)
            {
                const KernelSlot &s = kernelSlot(mode, bra.la, bra.lb, ket.la, ket.lb, v);
                if (!ownForm(v, s) || isF32Variant(v) != f32)
                    continue;
                const double t = variantTime(mode, bra, ket, s, f32, quartets, s.swap ? wavesKet : wavesBra);
                if (best < 0 || t < tBest)
                {
                    best = v;
                    tBest = t;
                }
            }
            if (ms)
                *ms = tBest;
            return best;
        }

        // Quartets of class pair (bra, ket) with lo <= Q_ab Q_cd < hi, from up to 64 evenly spaced
        // ket positions (both classes sorted by Q).
        double estimateQuartets(const PairClass &bra, const PairClass &ket, bool same, double lo, double hi)
        {
            if (bra.Qs.empty() || ket.Qs.empty())
                return double(bra.n_pairs) * ket.n_pairs * (same ? 0.5 : 1.0);
            const int samples = std::min(64, ket.n_pairs);
            double n = 0.0;
            for (int i = 0; i < samples; i++)
            {
                const double q = ket.Qs[static_cast<size_t>(i) * ket.n_pairs / samples];
                const int below = lo > 0 ? firstBelow(bra.Qs, q, lo) : bra.n_pairs;
                const int above = hi < kNoUpper ? firstBelow(bra.Qs, q, hi) : 0;
                n += std::max(0, below - above);
            }
            return n * ket.n_pairs / samples * (same ? 0.5 : 1.0);
        }

        // E matrices of a class interleaved over the lanes of each block of 64 lane positions
        // (KArgs::le): perm maps lane position -> position in order (null: the same)
        template <typename T>
        __global__ __launch_bounds__(256) void interleaveKernel(const T *__restrict__ in, T *__restrict__ out,
                                                                const int *order, const int *perm, const int *poff,
                                                                const int *pcnt, const long long *base, int n, int hs)
        {
            const int lane = threadIdx.x & 63;
            const int pos = 64 * static_cast<int>(blockIdx.x) + lane;
            const int pair = pos < n ? order[perm ? perm[pos] : pos] : -1;
            const T *src = pair >= 0 ? in + static_cast<size_t>(poff[pair]) * hs : in;
            const long long own = pair >= 0 ? static_cast<long long>(pcnt[pair]) * hs : 0;
            const long long rows = (base[blockIdx.x + 1] - base[blockIdx.x]) / 64;
            T *dst = out + base[blockIdx.x] + lane;
            for (long long r = 4LL * blockIdx.y + (threadIdx.x >> 6); r < rows; r += 4LL * gridDim.y)
                if (r < own)
                    dst[r * 64] = src[r];
        }

        __global__ void toFloatKernel(const double *__restrict__ in, float *__restrict__ out, long long n)
        {
            for (long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
                 i += static_cast<long long>(gridDim.x) * blockDim.x)
                out[i] = static_cast<float>(in[i]);
        }

        // FP32 copies b32, k32 of n doubles each; b32, whose presence says that both are there, last
        void toFloat(Context &c, const double *b, const double *k, float *&b32, float *&k32, long long n)
        {
            if (!k32)
                k32 = c.alloc<float>(n);
            float *out = c.alloc<float>(n);
            const int grid = static_cast<int>(std::min<long long>((n + 255) / 256, 65536));
            hipLaunchKernelGGL(toFloatKernel, dim3(grid), dim3(256), 0, c.stream, b, out, n);
            hipLaunchKernelGGL(toFloatKernel, dim3(grid), dim3(256), 0, c.stream, k, k32, n);
            LBX_HIP(hipGetLastError());
            b32 = out;
        }

        // FP32 copies of the E matrices, made once per context on first mixed-precision use
        void ensureF32(Context &c)
        {
            for (auto &pc : c.cls)
            {
                if (pc.d_eb32 || pc.n_ppairs == 0)
                    continue;
                toFloat(c, pc.d_eb, pc.d_ek, pc.d_eb32, pc.d_ek32, static_cast<long long>(pc.eCount()));
            }
        }

        // FP32 copies of the auxiliary shells' E matrices (mixed-precision RI sums)
        void ensureF32Aux(Context &c)
        {
            for (auto &pc : c.aux)
            {
                if (pc.d_eb32 || pc.n_ppairs == 0)
                    continue;
                toFloat(c, pc.d_eb, pc.d_ek, pc.d_eb32, pc.d_ek32, static_cast<long long>(pc.eCount()));
            }
        }

        // FP32 copies of the derivative E matrices (mixed-precision gradient)
        void ensureF32D1(Context &c)
        {
            for (auto &pc : c.cls)
            {
                if (pc.d_e1b32 || pc.n_ppairs == 0 || !pc.d_e1b)
                    continue;
                toFloat(c, pc.d_e1b, pc.d_e1k, pc.d_e1b32, pc.d_e1k32, 3 * static_cast<long long>(pc.eCount()));
            }
        }

        const KernelSlot &slotFor(int mode, const PairClass &bra, const PairClass &ket, int variant)
        {
            const KernelSlot &s = kernelSlot(mode, bra.la, bra.lb, ket.la, ket.lb, variant);
            if (!s.fn)
                throw Error(LBX_ERR_INVALID, "no kernel for class (" + std::to_string(bra.la) +
                                                     std::to_string(bra.lb) + "|" +
                                                     std::to_string(ket.la) + std::to_string(ket.lb) +
                                                     ") mode " + std::to_string(mode) + " variant " +
                                                     std::to_string(variant));
            return s;
        }

        // One launch of an unscreened driver: every (bra, ket) pair combination of a class pair
        struct PlainJob
        {
            int mode;
            const PairClass *bra, *ket;
            Pairing pairing;
            bool same;
            KArgs extra;
        };

        // Whether every pair of main shells has primitive pairs above the screen: the dense drivers
        // then write every element and need no zeroed output.
        bool allPairs(const Context &c)
        {
            size_t n = 0;
            for (const auto &pc : c.cls)
                n += pc.n_pairs;
            return n == c.shells.size() * (c.shells.size() + 1) / 2;
        }

        // One kernel of a call whose kernels are independent
        struct QueuedLaunch
        {
            Launcher fn;
            KArgs a;
            double cost;   // relative estimate of its time
        };

        // streams beside the context's that share the launches of one call (a process has four
        // hardware queues)
        constexpr int kSideStreams = SideStreams::kCount;

        // The independent launches of one call, spread over the context's stream and its side
        // streams: the side streams start after what the context's stream holds at construction
        // (fork event) and join() makes the context's stream wait for them.  Off (on = false):
        // everything on the context's stream.
        class Fan
        {
        public:
            Fan(SideStreams &side, hipStream_t main, bool on) : side_(side), main_(main), on_(on)
            {
                if (!on_)
                    return;
                side_.ensure();
                LBX_HIP(hipEventRecord(side_.fork, main_));
            }
            ~Fan()
            {
                // after an exception: still bring the side streams back to the context's stream
                for (int i = 0; i < kSideStreams; i++)
                    if (used_[i] && hipEventRecord(side_.joined[i], side_.s[i]) == hipSuccess)
                        (void)hipStreamWaitEvent(main_, side_.joined[i], 0);
            }
            Fan(const Fan &) = delete;
            Fan &operator=(const Fan &) = delete;

            // the least loaded stream
            hipStream_t pick(double cost)
            {
                int b = 0;
                if (on_)
                    for (int i = 1; i <= kSideStreams; i++)
                        if (load_[i] < load_[b])
                            b = i;
                load_[b] += cost;
                if (b == 0)
                    return main_;
                if (!used_[b - 1])
                {
                    LBX_HIP(hipStreamWaitEvent(side_.s[b - 1], side_.fork, 0));
                    used_[b - 1] = true;
                }
                return side_.s[b - 1];
            }

            void join()
            {
                for (int i = 0; i < kSideStreams; i++)
                    if (used_[i])
                    {
                        LBX_HIP(hipEventRecord(side_.joined[i], side_.s[i]));
                        LBX_HIP(hipStreamWaitEvent(main_, side_.joined[i], 0));
                        used_[i] = false;
                    }
            }

        private:
            SideStreams &side_;
            hipStream_t main_;
            bool on_;
            double load_[kSideStreams + 1] = {};
            bool used_[kSideStreams] = {};
        };

        // Launches the queue, most expensive first, over the fan's streams.
        void launchAll(std::vector<QueuedLaunch> &queue, Fan &fan)
        {
            std::stable_sort(queue.begin(), queue.end(),
                             [](const QueuedLaunch &x, const QueuedLaunch &y) { return x.cost > y.cost; });
            for (auto &l : queue)
            {
                l.fn(l.a, fan.pick(l.cost));
                LBX_HIP(hipGetLastError());
            }
            fan.join();
        }
    }

    KernelSlot &kernelSlot(int mode, int la, int lb, int lc, int ld, int variant)
    {
        static KernelSlot tab[N_MODES][kMaxLAux + 1][kMaxLMain + 1][kMaxLAux + 1][kMaxLMain + 1][N_VARIANTS];
        if (mode < 0 || mode >= N_MODES || la < 0 || la > kMaxLAux || lc < 0 || lc > kMaxLAux || lb < 0 ||
            lb > kMaxLMain || ld < 0 || ld > kMaxLMain || variant < 0 || variant >= N_VARIANTS)
            throw Error(LBX_ERR_INVALID, "kernel slot out of range");
        return tab[mode][la][lb][lc][ld][variant];
    }

    GradSlot &gradSlot(int la, int lb, int lc, int ld)
    {
        static GradSlot tab[kMaxLMain + 1][kMaxLMain + 1][kMaxLMain + 1][kMaxLMain + 1];
        if (la < 0 || la > kMaxLMain || lb < 0 || lb > kMaxLMain || lc < 0 || lc > kMaxLMain || ld < 0 ||
            ld > kMaxLMain)
            throw Error(LBX_ERR_INVALID, "gradient kernel slot out of range");
        return tab[la][lb][lc][ld];
    }

    // Algorithmic FLOPs of the gradient per quartet (7 ket-sized and 9 bra-sized transforms, R to
    // order L + 1, the density contraction of 12 derivative blocks), from a task table's sums.
    double gradFlops(const TaskTable &t, int la, int lb, int lc, int ld)
    {
        const double Hab = nHerm(la + lb), Hcd = nHerm(lc + ld);
        const double Sab = nSph(la) * nSph(lb), Scd = nSph(lc) * nSph(ld);
        return t.sum_kk * (7 * 2 * Hab * Hcd * Scd + rFlopsHost(la + lb + lc + ld + 1) + Hab * Hcd) +
               t.sum_kbra * 9 * 2 * Sab * Hab * Scd + t.quartets * 72 * Sab * Scd;
    }

    // Schwarz factors Q = sqrt(max |(ab|ab)|) of a class (computed on the device into d_q, pair
    // order) and the sorted order: by molecule, then Q descending (one molecule in an ordinary
    // context), so that each ket's surviving bra pairs form a prefix and each molecule's pairs
    // keep their contiguous range of positions.
    void sortByBound(PairClass &pc)
    {
        if (pc.n_pairs == 0)
            return;
        pc.Q.resize(pc.n_pairs);
        LBX_HIP(hipMemcpy(pc.Q.data(), pc.d_q, pc.n_pairs * sizeof(double), hipMemcpyDeviceToHost));
        std::vector<int> order(pc.n_pairs);
        std::iota(order.begin(), order.end(), 0);
        std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
            return pc.mol[x] != pc.mol[y] ? pc.mol[x] < pc.mol[y] : pc.Q[x] > pc.Q[y];
        });
        std::vector<double> qs(pc.n_pairs);
        for (int i = 0; i < pc.n_pairs; i++)
            qs[i] = pc.Q[order[i]];
        pc.order = order;
        pc.Qs = qs;
        // the longest primitive loop of each 64-pair block, in the count order of lanePerm
        std::vector<int> count(pc.n_pairs), none(pc.n_pairs, 0);
        for (int i = 0; i < pc.n_pairs; i++)
            count[i] = -pc.pcnt[order[i]];
        const tasks::LaneOrder lo = tasks::laneOrder(qs, count, none);
        double kl = 0.0;
        for (int b = 0; b < pc.n_pairs; b += 64)
        {
            int m = 0;
            for (int i = b; i < std::min(b + 64, pc.n_pairs); i++)
                m = std::max(m, -count[lo.perm[i]]);
            kl += m;
        }
        pc.klane = kl / ((pc.n_pairs + 63) / 64);
        LBX_HIP(hipMemcpy(pc.d_order, order.data(), order.size() * sizeof(int), hipMemcpyHostToDevice));
        LBX_HIP(hipMemcpy(pc.d_q, qs.data(), qs.size() * sizeof(double), hipMemcpyHostToDevice));
    }
}

using namespace lbx;

struct lbx_context : Context
{
    // J/K task tables per (bra class, ket class, bound range [lo, hi), variant); Q does not
    // depend on D
    std::map<std::tuple<int, int, double, double, int>, TaskTable> jk_tasks;
    // kernel variant per class pair chosen by lbx_tune (absent: work-estimate default), for
    // the FP64 build and for the FP32 tier of the mixed build
    std::map<std::pair<int, int>, int> tuned, tuned32;
    // lbx_set_class_filter: the one class pair (bra class, ket class) lbx_jk evaluates; -1: all
    int filter_i = -1, filter_j = -1;
    // lbx_set_graphs: capture the J/K launch sequences and the RI sums into HIP graphs and
    // replay them (off by default: a capture in progress makes synchronous HIP calls of other
    // threads on the legacy stream fail)
    bool graphs = false;
    // lbx_set_bound_window: lbx_jk evaluates only quartets with window_lo <= Q_ab Q_cd < window_hi
    double window_lo = 0.0, window_hi = kNoUpper;
    SideStreams side;
    // task tables of the unscreened drivers per (lane class, uniform class, pairing, same, width)
    std::map<std::tuple<const PairClass *, const PairClass *, int, bool, int>, TaskTable> plain_tasks;

    // Runs the jobs (independent of each other) over the context's streams and waits for them.
    void runPlain(const std::vector<PlainJob> &jobs)
    {
        std::vector<QueuedLaunch> queue;
        for (const PlainJob &job : jobs)
        {
            const PairClass &bra = *job.bra, &ket = *job.ket;
            if (bra.n_pairs == 0 || ket.n_pairs == 0)
                continue;
            // tasks of a one-lane form: per uniform-side pair, its lane-side pairs in blocks of 64
            const double nb = bra.n_pairs, nk = ket.n_pairs, half = job.same ? 0.5 : 1.0;
            const bool diag = job.pairing == Pairing::Diagonal;
            double ms = 0.0;
            const int var = defaultVariant(job.mode, bra, ket, false, diag ? nb : half * nb * nk,
                                           diag ? nb : nk * std::ceil(half * nb / 64), 0.0, &ms);
            const KernelSlot &s = slotFor(job.mode, bra, ket, var);
            const auto key = std::make_tuple(&bra, &ket, static_cast<int>(job.pairing), job.same, s.width);
            auto it = plain_tasks.find(key);
            if (it == plain_tasks.end())
                it = plain_tasks.emplace(key, buildTasks(*this, bra, ket, job.pairing, job.same, 0.0, s.width)).first;
            KArgs a = baseArgs(*this, bra, ket, it->second, job.same);
            a.out = job.extra.out;
            a.kind = job.extra.kind;
            a.qout = job.extra.qout;
            a.dout = job.extra.dout;
            queue.push_back({s.fn, a, ms});
        }
        flushStaged();
        Fan fan(side, stream, queue.size() > 1);
        launchAll(queue, fan);
        LBX_HIP(hipStreamSynchronize(stream));
    }

    // Schwarz factors and sorted order of every main class (kind 4: pairs) or auxiliary class
    // (kind 2: single shells)
    void sortAll(std::vector<PairClass> &classes, int kind)
    {
        std::vector<PlainJob> jobs;
        for (auto &pc : classes)
        {
            KArgs extra{};
            extra.qout = pc.d_q;
            extra.kind = kind;
            jobs.push_back({MODE_DIAG, &pc, &pc, Pairing::Diagonal, true, extra});
        }
        runPlain(jobs);
        for (auto &pc : classes)
            sortByBound(pc);
    }

    void ensureSchwarz()
    {
        if (have_schwarz)
            return;
        sortAll(cls, 4);
        have_schwarz = true;
    }

    // the same for the auxiliary shells (bounds of the RI sums' precision split)
    void ensureSchwarzAux()
    {
        if (have_schwarz_aux)
            return;
        sortAll(aux, 2);
        have_schwarz_aux = true;
    }

    // lbx_eri*_batch: (shell a, shell b) -> pair index per main pair class
    std::vector<std::unordered_map<long long, int>> pair_maps;
    // their task list on the device (1 MiB, made on first use; every call waits for its kernel)
    static constexpr size_t kBlockTaskInts = 1 << 18;
    int *block_tasks = nullptr;
    // this device's scratch array (lbx_eri4_batch_static)
    int *d_scratch = nullptr;

    // the default forms, per class pair, bound range and tier, with their estimated times
    struct Choice
    {
        int variant;
        double ms;
    };
    std::map<std::tuple<int, int, double, double, bool>, Choice> defaults;

    Choice defaultFor(int i, int j, double lo, double hi, bool f32)
    {
        const auto key = std::make_tuple(i, j, lo, hi, f32);
        auto it = defaults.find(key);
        if (it == defaults.end())
        {
            const double n = estimateQuartets(cls[i], cls[j], i == j, lo, hi);
            Choice ch{-1, 0.0};
            ch.variant = defaultVariant(MODE_JK, cls[i], cls[j], f32, n, std::max(1.0, n / 64), std::max(1.0, n / 64), &ch.ms);
            it = defaults.emplace(key, ch).first;
        }
        return it->second;
    }

    // form of the FP64 quartets of class pair (i, j) with bounds in [lo, hi)
    int variantFor(int i, int j, double lo, double hi)
    {
        auto it = tuned.find({i, j});
        return it != tuned.end() ? it->second : defaultFor(i, j, lo, hi, false).variant;
    }

    // form of the small-bound quartets of a mixed build: an FP32 form, or an FP64 one
    // where the class has no FP32 form or tuning found the FP64 form faster
    int variant32For(int i, int j, double lo, double hi)
    {
        auto it = tuned32.find({i, j});
        if (it != tuned32.end())
            return it->second;
        const int v = defaultFor(i, j, lo, hi, true).variant;
        return v >= 0 ? v : variantFor(i, j, lo, hi);
    }

    // Lane side of the one-lane J/K kernels, per pair class: Schwarz-order positions regrouped
    // within half-decade buckets of the Schwarz factor (lane position -> Schwarz-order position),
    // and the range of Schwarz-order positions each 64-lane block holds.  Regrouped by primitive
    // count when the kernel sums K in LDS, so that a wave's lanes run loops of one length; else by
    // shell, so that lanes sharing the first shell are adjacent and combine their K updates.
    struct LanePerm
    {
        std::vector<int> perm, bqlo, bqhi;
        int *d_perm = nullptr, *d_bqlo = nullptr, *d_bqhi = nullptr;
    };
    std::map<std::pair<int, bool>, LanePerm> lane_perm;

    const LanePerm &lanePerm(int idx, bool byCount)
    {
        auto it = lane_perm.find({idx, byCount});
        if (it != lane_perm.end())
            return it->second;
        const PairClass &pc = cls[idx];
        const int n = pc.n_pairs;
        std::vector<double> qs(n);
        std::vector<int> sa(n), sb(n);
        for (int p = 0; p < n; p++)
        {
            qs[p] = pc.Q.empty() ? 1.0 : pc.Q[pc.order[p]];
            // longest primitive loops first
            sa[p] = byCount ? -pc.pcnt[pc.order[p]] : pc.sh_a[pc.order[p]];
            sb[p] = byCount ? 0 : pc.sh_b[pc.order[p]];
        }
        tasks::LaneOrder lo = tasks::laneOrder(qs, sa, sb);
        LanePerm lp;
        std::vector<int> perm = std::move(lo.perm);
        lp.bqlo = std::move(lo.bqlo);
        lp.bqhi = std::move(lo.bqhi);
        lp.d_perm = stage(perm);
        lp.d_bqlo = stage(lp.bqlo);
        lp.d_bqhi = stage(lp.bqhi);
        lp.perm = std::move(perm);
        return lane_perm.emplace(std::make_pair(idx, byCount), std::move(lp)).first->second;
    }

    // Lane-interleaved E matrices (KArgs::le) per lane order and use (bra or ket).  The orders are
    // made after the Schwarz order, which stays for the context's life.
    struct LaneE
    {
        long long *base = nullptr;
        double *e = nullptr;
        float *e32 = nullptr;
    };
    std::map<std::pair<const LanePerm *, bool>, LaneE> lane_e;

    // Device memory that only saves time: the interleaved copies of E and the parts of J.  At most a
    // quarter of the device's; where there is no room for one, the call takes forms that need none,
    // and a call that runs out of memory frees them all and is made again without (guardedIn).
    std::vector<void *> extras;
    size_t extra_bytes = 0, extra_cap = 0;
    bool no_extras = false;   // after such a call
    bool capturing = false;   // a capture allocates nothing: it takes what the eager call before it took

    template <class T>
    T *takeExtra(size_t n)
    {
        if (no_extras || capturing)
            return nullptr;
        if (extra_cap == 0)
        {
            size_t total = 0;
            LBX_HIP(hipDeviceTotalMem(&total, device));
            extra_cap = total / 4;
        }
        const size_t bytes = std::max<size_t>(n, 1) * sizeof(T);
        void *p = extra_bytes + bytes <= extra_cap ? take(bytes) : nullptr;
        if (p)
        {
            extras.push_back(p);
            extra_bytes += bytes;
        }
        return static_cast<T *>(p);
    }

    // Frees them (between calls) with the graphs and launches that were made with them.
    bool freeExtras()
    {
        if (extras.empty())
            return false;
        LBX_HIP(hipStreamSynchronize(stream));
        dropJKGraphs();
        dropRiGraph();
        ri_prepared.clear();
        ri_launches.clear();
        for (auto &kv : lane_e)
            kv.second.e = nullptr, kv.second.e32 = nullptr;
        for (auto &kv : sum_e)
            kv.second.e = nullptr, kv.second.e32 = nullptr;
        j_parts = nullptr;
        for (void *p : extras)
            giveBack(p);
        extras.clear();
        extra_bytes = 0;
        return true;
    }

    // The interleaved E of a lane side, made on first use; false when there is no room for it.
    bool interleave(LaneE &le, const PairClass &pc, bool ket, const std::vector<int> &order,
                    const std::vector<int> *perm, const int *d_order, const int *d_perm, bool f32)
    {
        if (f32 ? le.e32 != nullptr : le.e != nullptr)
            return true;
        if (capturing)
            return false;
        const int hs = nHerm(pc.la + pc.lb) * nSph(pc.la) * nSph(pc.lb), nblk = (pc.n_pairs + 63) / 64;
        std::vector<long long> base(nblk + 1, 0);
        for (int b = 0; b < nblk; b++)
        {
            int k = 0;
            for (int p = 64 * b; p < std::min(64 * b + 64, pc.n_pairs); p++)
                k = std::max(k, pc.pcnt[order[perm ? (*perm)[p] : p]]);
            base[b + 1] = base[b] + 64LL * k * hs;
        }
        float *e32 = f32 ? takeExtra<float>(base[nblk]) : nullptr;
        double *e = f32 ? nullptr : takeExtra<double>(base[nblk]);
        if (!e && !e32)
            return false;
        if (!le.base)
            le.base = upload(base);
        flushStaged();   // the orders
        const dim3 grid(nblk, 16);
        auto run = [&](auto *out, auto *in) {
            using T = std::remove_reference_t<decltype(*out)>;
            hipLaunchKernelGGL(interleaveKernel<T>, grid, dim3(256), 0, stream, in, out, d_order, d_perm, pc.d_poff,
                               pc.d_pcnt, le.base, pc.n_pairs, hs);
            LBX_HIP(hipGetLastError());
        };
        if (f32)
        {
            run(e32, ket ? pc.d_ek32 : pc.d_eb32);
            le.e32 = e32;
        }
        else
        {
            run(e, ket ? pc.d_ek : pc.d_eb);
            le.e = e;
        }
        return true;
    }

    // Pair order of the RI sums without a bound range: by molecule, then the longest primitive
    // loops first.  Unlike the classes' order it does not change when the Schwarz factors are made,
    // so launches prepared before that stay good.
    struct SumOrder
    {
        std::vector<int> order;
        int *d_order = nullptr;
    };
    std::map<const PairClass *, SumOrder> sum_orders;
    // the lane sides' interleaved E in that order or (true) in the Schwarz order
    std::map<std::pair<const PairClass *, bool>, LaneE> sum_e;

    const SumOrder &sumOrder(const PairClass &pc)
    {
        SumOrder &so = sum_orders[&pc];
        if (!so.d_order)
        {
            so.order = pc.order;
            std::stable_sort(so.order.begin(), so.order.end(), [&](int x, int y) {
                return pc.mol[x] != pc.mol[y] ? pc.mol[x] < pc.mol[y] : pc.pcnt[x] > pc.pcnt[y];
            });
            so.d_order = stage(so.order);
        }
        return so;
    }

    // whether the lane side's E of a one-lane RI sum launch is there
    bool sumLaneReady(const PairClass &lane, bool bounded, bool f32)
    {
        const std::vector<int> &order = bounded ? lane.order : sumOrder(lane).order;
        return interleave(sum_e[{&lane, bounded}], lane, false, order, nullptr, bounded ? lane.d_order : sumOrder(lane).d_order,
                          nullptr, f32);
    }

    // orders and (one-lane forms, sumLaneReady) the lane side's E of an RI sum launch
    void setSumSides(KArgs &a, const PairClass &lane, const PairClass &unif, bool bounded, int kind)
    {
        if (!bounded)
        {
            a.bra.order = sumOrder(lane).d_order;
            a.ket.order = sumOrder(unif).d_order;
        }
        if (kind != KIND_LANE)
            return;
        const LaneE &le = sum_e[{&lane, bounded}];
        a.le = le.e;
        a.le32 = le.e32;
        a.lbase = le.base;
    }

    // Columns of the K rows that the one-lane kernels sum in LDS, per lane-side class: the functions
    // of its shells' angular momenta (KArgs::kcol_a ..)
    struct KCols
    {
        int *d_a = nullptr, *d_b = nullptr, *d_ao = nullptr;
        int n = 0;
    };
    std::map<int, KCols> k_cols;

    int kColumns(const PairClass &pc) const
    {
        int n = 0;
        for (const auto &s : shells)
            n += (s.l == pc.la || s.l == pc.lb) ? nSph(s.l) : 0;
        return n;
    }

    const KCols &kCols(int idx)
    {
        auto it = k_cols.find(idx);
        if (it != k_cols.end())
            return it->second;
        const PairClass &pc = cls[idx];
        std::vector<int> col(shells.size(), 0), ao, a(pc.n_pairs), b(pc.n_pairs);
        for (int l : {pc.la, pc.lb})
        {
            for (size_t s = 0; s < shells.size(); s++)
                if (shells[s].l == l)
                {
                    col[s] = static_cast<int>(ao.size());
                    for (int m = 0; m < nSph(l); m++)
                        ao.push_back(static_cast<int>(shells[s].ao) + m);
                }
            if (pc.la == pc.lb)
                break;
        }
        for (int p = 0; p < pc.n_pairs; p++)
        {
            a[p] = col[pc.sh_a[p]];
            b[p] = col[pc.sh_b[p]];
        }
        KCols k;
        k.d_a = stage(a);
        k.d_b = stage(b);
        k.d_ao = stage(ao);
        k.n = static_cast<int>(ao.size());
        return k_cols.emplace(idx, k).first->second;
    }

    // The lane side of a one-lane J/K kernel
    struct JKLane
    {
        const LanePerm *lp = nullptr;
        const LaneE *le = nullptr;
        bool kLds = false;   // K rows of the uniform pair in LDS
    };

    // false when there is no room for its interleaved E
    bool jkLane(int i, int j, const KernelSlot &s, bool f32, JKLane &l)
    {
        const PairClass &lside = s.swap ? cls[j] : cls[i], &uside = s.swap ? cls[i] : cls[j];
        // K rows of the uniform pair in LDS: up to 64 KiB, and at least three lane blocks to share
        // them (a workgroup's four waves take four blocks of a group); else K by atomics alone, which
        // bound the classes of low angular momentum (16 updates per (ps|ps) quartet at 23 G/s:
        // (H2O)10 def2-TZVP (ps|ps) 2.3 ms, with the rows in LDS 1.1)
        l.kLds = lside.n_pairs > 128 && (nSph(uside.la) + nSph(uside.lb)) * kColumns(lside) * 8 <= 65536;
        l.lp = &lanePerm(s.swap ? j : i, l.kLds);
        LaneE &le = lane_e[{l.lp, s.swap}];
        l.le = &le;
        return interleave(le, lside, s.swap, lside.order, &l.lp->perm, lside.d_order, l.lp->d_perm, f32);
    }

    // The J/K kernel of class pair (i >= j) with the given variant (the one-wave form in its place
    // when the one-lane form is not built or its copy of E has no room), its arguments over the quartets with
    // lo <= Q_ab Q_cd < hi (staged tables: flushStaged() before the launch) and its task table.
    struct JKLaunch
    {
        Launcher fn;
        KArgs a;
        const TaskTable *t;
        int var;
    };
    JKLaunch prepareJK(int i, int j, int var, const double *D, double *J, double *K,
                       double thresh, double thresh_hi = kNoUpper)
    {
        const PairClass &bra = cls[i], &ket = cls[j];
        // the number of the form that runs, which the profile reports
        JKLane lane;
        const KernelSlot &asked = slotFor(MODE_JK, bra, ket, var);
        if (!ownForm(var, asked) || (asked.kind == KIND_LANE && !jkLane(i, j, asked, isF32Variant(var), lane)))
            var = isF32Variant(var) ? VAR_MFMA32 : VAR_MFMA;
        const KernelSlot &s = slotFor(MODE_JK, bra, ket, var);
        // the one-wave-per-quartet kernel walks consecutive tasks of one pair of the side whose
        // E matrices are larger, so those stay in cache across the tasks
        auto eBytes = [](const PairClass &c)
        { return c.n_pairs ? double(c.n_ppairs) / c.n_pairs * nHerm(c.la + c.lb) * nSph(c.la) * nSph(c.lb) : 0.0; };
        const bool braMajor = !s.swap && s.kind == KIND_WAVE && i != j && eBytes(bra) > eBytes(ket);
        // the block kernel's tasks: per bra position, blocks of s.width consecutive ket positions
        const bool blockKind = s.kind == KIND_BLOCK;
        const auto key = std::make_tuple(i, j, thresh, thresh_hi, var);
        auto it = jk_tasks.find(key);
        if (it == jk_tasks.end())
            it = jk_tasks
                         .emplace(key, (s.swap || braMajor || blockKind)
                                               ? buildTasks(*this, ket, bra, Pairing::Unique, blockKind && i == j,
                                                            thresh, s.width, false, thresh_hi)
                                               : buildTasks(*this, bra, ket, Pairing::Unique, i == j, thresh,
                                                            s.width, true, thresh_hi))
                         .first;
        // The one-lane-per-quartet kernels run their tasks by groups of lane blocks: as many
        // blocks (a power of two, up to 64) as keep the lane side's E matrices of a group within
        // about 1 MiB of L2, so each uniform pair's E is read once per group.
        const bool blockMajor = s.kind == KIND_LANE;
        const PairClass &lside = s.swap ? ket : bra;
        const int nlane = lside.n_pairs;
        int gshift = 0;
        if (blockMajor)
        {
            const double groupBytes = 64.0 * eBytes(lside) * (isF32Variant(var) ? 4 : 8);
            while (gshift < 6 && groupBytes * (2 << gshift) <= double(1 << 20))
                gshift++;
        }
        const LanePerm *lp = lane.lp;
        if (blockMajor && lane.kLds)
            gshift = std::max(gshift, 2);
        if (blockMajor && it->second.nblk == 0)
            buildBlockMajor(*this, it->second, nlane, 1, gshift, lp->perm, lp->bqlo, lp->bqhi);
        const TaskTable &t = it->second;
        KArgs a = baseArgs(*this, bra, ket, t, i == j);
        a.bra_major = braMajor ? 1 : 0;
        a.D = D;
        a.J = J;
        a.K = K;
        if (blockMajor && t.nblk > 0)
        {
            a.block_major = 1;
            a.nblk = t.nblk;
            a.gshift = t.gshift;
            a.lperm = lp->d_perm;
            a.bqlo = lp->d_bqlo;
            a.bqhi = lp->d_bqhi;
            a.bprefix = t.d_bprefix;
            a.bq0 = t.d_bq0;
            a.ntasks = t.btasks;
            a.le = lane.le->e;
            a.le32 = lane.le->e32;
            a.lbase = lane.le->base;
            if (lane.kLds)
            {
                const KCols &k = kCols(s.swap ? j : i);
                a.kcol_a = k.d_a;
                a.kcol_b = k.d_b;
                a.kao = k.d_ao;
                a.kcols = k.n;
            }
        }
        if (sample_quartets > 0 && a.block_major)
        {
            // every stride-th lane block with all its uniform-side partners
            auto st = tune_tasks.find(key);
            if (st == tune_tasks.end())
            {
                const int stride = static_cast<int>(
                        std::max(1.0, std::ceil(t.quartets / static_cast<double>(sample_quartets))));
                TaskTable ts;
                ts.nket = t.nket;
                ts.plo = t.plo;
                ts.phi = t.phi;
                ts.cuts = t.cuts;
                ts.quartets = buildBlockMajor(*this, ts, nlane, stride, t.gshift, lp->perm, lp->bqlo, lp->bqhi);
                st = tune_tasks.emplace(key, std::move(ts)).first;
            }
            const TaskTable &ts = st->second;
            a.bprefix = ts.d_bprefix;
            a.bq0 = ts.d_bq0;
            a.ntasks = ts.btasks;
            sampled = ts.quartets;
        }
        else if (sample_quartets > 0)
        {
            // every stride-th uniform-side position, about sample_quartets quartets spread over
            // the whole range of Schwarz bounds
            auto st = tune_tasks.find(key);
            if (st == tune_tasks.end())
            {
                const int stride = static_cast<int>(
                        std::max(1.0, std::ceil(t.quartets / static_cast<double>(sample_quartets))));
                TaskTable ts;
                ts.nket = t.nket;
                ts.plo = t.plo;
                ts.phi = t.phi;
                ts.prefix.resize(t.nket + 1);
                long long acc = 0;
                for (int q = 0; q < t.nket; q++)
                {
                    if (q % stride != 0)
                        ts.phi[q] = ts.plo[q];
                    ts.prefix[q] = acc;
                    const long long cnt = ts.phi[q] - ts.plo[q];
                    acc += (cnt + s.width - 1) / s.width;
                    ts.quartets += static_cast<double>(cnt);
                }
                ts.prefix[t.nket] = acc;
                ts.ntasks = acc;
                ts.d_prefix = stage(ts.prefix);
                ts.d_plo = stage(ts.plo);
                ts.d_phi = stage(ts.phi);
                st = tune_tasks.emplace(key, std::move(ts)).first;
            }
            const TaskTable &ts = st->second;
            a.prefix = ts.d_prefix;
            a.plo = ts.d_plo;
            a.phi = ts.d_phi;
            a.ntasks = ts.ntasks;
            sampled = ts.quartets;
        }
        return {s.fn, a, &t, var};
    }

    // Queues it on the context stream; returns the variant that runs.
    int launchJK(int i, int j, int var, const double *D, double *J, double *K, double thresh)
    {
        const JKLaunch l = prepareJK(i, j, var, D, J, K, thresh);
        flushStaged();
        l.fn(l.a, stream);
        LBX_HIP(hipGetLastError());
        return l.var;
    }

    // when > 0, launchJK runs only a sample of ~sample_quartets quartets (autotuner timing) and
    // leaves their count in `sampled`
    long long sample_quartets = 0;
    double sampled = 0;
    std::map<std::tuple<int, int, double, double, int>, TaskTable> tune_tasks;   // the samples

    // gradient task tables per (bra class, ket class, Schwarz threshold)
    std::map<std::tuple<int, int, double, double>, TaskTable> grad_tasks;

    // batched RI sums: the whole launch sequence captured once into a graph (per output buffer)
    hipGraph_t ri_graph = nullptr;
    hipGraphExec_t ri_exec = nullptr;
    double *ri_out = nullptr;
    double ri_triplets = 0, ri_doublets = 0, ri_flops = 0, ri_triplets32 = 0, ri_doublets32 = 0;
    double ri_split = 0.0;   // precision split the prepared launches were built for (0: FP64)

    void dropRiGraph()
    {
        if (ri_exec)
            (void)hipGraphExecDestroy(ri_exec);
        if (ri_graph)
            (void)hipGraphDestroy(ri_graph);
        ri_exec = nullptr;
        ri_graph = nullptr;
        ri_out = nullptr;
    }

    // Kernel launches of the RI sums: every eri3 (pair class | aux l) and eri2
    // (aux l | aux l' <= l) class pair, with task tables built once per precision split (device
    // memory cannot be allocated while a stream is being captured).  split > 0: the triplets and
    // doublets with bound Q_ab Q_P below it in the FP32 form where the class has one.
    std::vector<QueuedLaunch> ri_launches;
    std::map<double, std::vector<QueuedLaunch>> ri_prepared;
    std::map<double, std::array<double, 5>> ri_counts;   // triplets, doublets, flops, FP32 ones
    // FP64 variant of each RI class pair chosen by lbx_tune on a batched context, keyed by
    // (kind, lane class, uniform class): kind 3 (main pair class | aux l), 2 (aux l | aux l')
    std::map<std::tuple<int, int, int>, int> tuned_sum;

    int sumVariant(int kind, int il, int iu, const PairClass &lane, const PairClass &unif) const
    {
        auto it = tuned_sum.find({kind, il, iu});
        if (it != tuned_sum.end())
            return it->second;
        // pairs per molecule on each side
        std::vector<int> nl(nmol, 0), nu(nmol, 0);
        for (int m : lane.mol)
            nl[m]++;
        for (int m : unif.mol)
            nu[m]++;
        double quartets = 0.0, waves = 0.0;
        const double half = kind == 2 && il == iu ? 0.5 : 1.0;
        for (int m = 0; m < nmol; m++)
        {
            quartets += half * nl[m] * nu[m];
            waves += nu[m] * std::ceil(half * nl[m] / 64);
        }
        return defaultVariant(MODE_SUM, lane, unif, false, quartets, waves, 0.0);
    }

    // Times the FP64 sum kernels of every RI class pair (the one-lane form and the MFMA form,
    // each over the class pair's whole task table into a scratch output) and keeps the faster.
    void tuneRiSums()
    {
        DevBuf scratch(4LL * nmol);
        hipEvent_t e0, e1;
        LBX_HIP(hipEventCreate(&e0));
        LBX_HIP(hipEventCreate(&e1));
        auto one = [&](int kind, int il, int iu, const PairClass &lane, const PairClass &unif, bool same)
        {
            if (lane.n_pairs == 0 || unif.n_pairs == 0)
                return;
            int best = -1;
            float best_ms = 0.0f;
            for (int v : {static_cast<int>(VAR_VALU_BRA), static_cast<int>(VAR_MFMA)})
            {
                const KernelSlot &k = kernelSlot(MODE_SUM, lane.la, lane.lb, unif.la, unif.lb, v);
                if (!k.fn || (k.kind == KIND_LANE && !sumLaneReady(lane, false, false)))
                    continue;
                TaskTable t = buildTasksMol(*this, lane, unif, same, k.width, 0.0, kNoUpper, false);
                KArgs a = baseArgs(*this, lane, unif, t, same);
                a.kind = kind;
                a.out = scratch.p;
                setSumSides(a, lane, unif, false, k.kind);
                flushStaged();
                k.fn(a, stream);   // loads the code
                LBX_HIP(hipEventRecord(e0, stream));
                k.fn(a, stream);
                LBX_HIP(hipEventRecord(e1, stream));
                LBX_HIP(hipGetLastError());
                LBX_HIP(hipEventSynchronize(e1));
                float ms = 0.0f;
                LBX_HIP(hipEventElapsedTime(&ms, e0, e1));
                if (best < 0 || ms < best_ms)
                {
                    best = v;
                    best_ms = ms;
                }
                // the table's device arrays were allocated from the context; free them now
                for (void *p : {static_cast<void *>(t.d_prefix), static_cast<void *>(t.d_plo),
                                static_cast<void *>(t.d_phi), static_cast<void *>(t.d_bprefix),
                                static_cast<void *>(t.d_bq0)})
                    giveBack(p);
            }
            if (best >= 0)
                tuned_sum[{kind, il, iu}] = best;
        };
        try
        {
            for (int i = 0; i < static_cast<int>(cls.size()); i++)
                for (int l = 0; l < static_cast<int>(aux.size()); l++)
                    one(3, i, l, cls[i], aux[l], false);
            for (int la = 0; la < static_cast<int>(aux.size()); la++)
                for (int lc = 0; lc <= la; lc++)
                    one(2, la, lc, aux[la], aux[lc], la == lc);
        }
        catch (...)
        {
            (void)hipEventDestroy(e0);
            (void)hipEventDestroy(e1);
            throw;
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        freeExtras();   // the forms that lost keep nothing
        dropRiGraph();
        ri_prepared.clear();
        ri_counts.clear();
    }

    void prepareRiSums(double split)
    {
        auto it = ri_prepared.find(split);
        if (it == ri_prepared.end())
        {
            std::vector<QueuedLaunch> launches;
            std::array<double, 5> n{0, 0, 0, 0, 0};
            auto add = [&](const PairClass &lane, const PairClass &unif, bool same, int kind, int il, int iu)
            {
                if (lane.n_pairs == 0 || unif.n_pairs == 0)
                    return;
                const int var = sumVariant(kind, il, iu, lane, unif);
                const KernelSlot &ks = slotFor(MODE_SUM, lane, unif, var);
                const KernelSlot &k32 = kernelSlot(MODE_SUM, lane.la, lane.lb, unif.la, unif.lb, VAR_VALU_BRA32);
                const bool tiers = split > 0.0 && k32.fn;
                auto one = [&](const KernelSlot &form, double lo, double hi, bool fp32)
                {
                    // without room for the copy of E, the one-wave form (FP64)
                    const bool room = form.kind != KIND_LANE || sumLaneReady(lane, split > 0.0, fp32);
                    const KernelSlot &k = room ? form : slotFor(MODE_SUM, lane, unif, VAR_MFMA);
                    fp32 = fp32 && room;
                    TaskTable t = buildTasksMol(*this, lane, unif, same, k.width, lo, hi);
                    KArgs a = baseArgs(*this, lane, unif, t, same);
                    a.kind = kind;
                    setSumSides(a, lane, unif, split > 0.0, k.kind);
                    launches.push_back({k.fn, a, variantTime(MODE_SUM, lane, unif, k, fp32, t.quartets, double(t.ntasks))});
                    n[kind == 3 ? 0 : 1] += t.quartets;
                    n[2] += t.flops;
                    if (fp32)
                        n[kind == 3 ? 3 : 4] += t.quartets;
                };
                if (tiers)
                {
                    one(ks, split, kNoUpper, false);
                    one(k32, 0.0, split, true);
                }
                else
                    one(ks, 0.0, kNoUpper, false);
            };
            for (int i = 0; i < static_cast<int>(cls.size()); i++)
                for (int l = 0; l < static_cast<int>(aux.size()); l++)
                    add(cls[i], aux[l], false, 3, i, l);
            for (int la = 0; la < static_cast<int>(aux.size()); la++)
                for (int lc = 0; lc <= la; lc++)
                    add(aux[la], aux[lc], la == lc, 2, la, lc);
            flushStaged();
            it = ri_prepared.emplace(split, std::move(launches)).first;
            ri_counts[split] = n;
        }
        ri_launches = it->second;
        const auto &n = ri_counts[split];
        ri_triplets = n[0];
        ri_doublets = n[1];
        ri_flops = n[2];
        ri_triplets32 = n[3];
        ri_doublets32 = n[4];
    }

    // fill + launches on stream s (the capture stream)
    void queueRiSums(double *out, hipStream_t s)
    {
        fill(out, 4LL * nmol, 0.0, s);
        std::vector<QueuedLaunch> queue = ri_launches;
        for (auto &l : queue)
            l.a.out = out;
        Fan fan(side, s, queue.size() > 1);
        launchAll(queue, fan);
    }

    // The gradient kernel of class pair (i >= j) over the quartets with
    // thresh <= Q_ab Q_cd < thresh_hi, in FP32 arithmetic when fp32.
    struct GradLaunch
    {
        GradLauncher fn;
        GArgs a;
        const TaskTable *t;
    };
    // parts of J besides the caller's matrix (queueJK)
    double *j_parts = nullptr;
    // gradients the kernels' workgroups add to (GArgs::grad), summed at the end
    static constexpr int kGradCopies = 64;
    double *grad_copies = nullptr;

    GradLaunch prepareGrad(int i, int j, const double *D, double thresh,
                           double thresh_hi = kNoUpper, bool fp32 = false)
    {
        const PairClass &ci = cls[i], &cj = cls[j];
        const bool lane_i = gradLaneFirst(ci.la, ci.lb, cj.la, cj.lb);
        const PairClass &lane = lane_i ? ci : cj, &unif = lane_i ? cj : ci;
        const GradSlot &s = gradSlot(lane.la, lane.lb, unif.la, unif.lb);
        if (!s.fn || !s.fn32)
            throw Error(LBX_ERR_INVALID, "no gradient kernel for this class pair");
        const auto key = std::make_tuple(i, j, thresh, thresh_hi);
        auto it = grad_tasks.find(key);
        if (it == grad_tasks.end())
            it = grad_tasks
                         .emplace(key, buildTasks(*this, lane, unif, Pairing::Unique, i == j, thresh, s.width,
                                                  lane_i, thresh_hi))
                         .first;
        const TaskTable &t = it->second;
        GArgs a{};
        a.lane = lane.view();
        a.unif = unif.view();
        a.prefix = t.d_prefix;
        a.plo = t.d_plo;
        a.phi = t.d_phi;
        a.nket = t.nket;
        a.ntasks = t.ntasks;
        a.same_class = i == j ? 1 : 0;
        a.boys = d_boys;
        a.D = D;
        a.nbf = static_cast<long long>(nbf);
        a.grad = grad_copies;
        a.ncopy = kGradCopies;
        a.stride = 3LL * natoms;
        return {fp32 ? s.fn32 : s.fn, a, &t};
    }

    // Queues one J/K build on the context stream: J and K cleared, every class pair's kernel
    // (the FP32 tier of a mixed build below `split`), J and K symmetrised.
    lbx_jk_stats queueJK(const double *D, double *J, double *K, double schwarz_thresh, double split,
                         bool mixed, bool prof_on);

    // J/K launch sequences captured into graphs, per (D, J, K, Schwarz threshold, split, mixed);
    // dropped when the variant choice changes (lbx_tune, lbx_set_variant)
    using JKKey = std::tuple<const double *, double *, double *, double, double, int>;
    struct JKGraph
    {
        hipGraph_t graph = nullptr;
        hipGraphExec_t exec = nullptr;
        lbx_jk_stats stats{};
    };
    std::map<JKKey, JKGraph> jk_graphs;
    static constexpr size_t kMaxJKGraphs = 8;

    void dropJKGraphs()
    {
        for (auto &kv : jk_graphs)
        {
            if (kv.second.exec)
                (void)hipGraphExecDestroy(kv.second.exec);
            if (kv.second.graph)
                (void)hipGraphDestroy(kv.second.graph);
        }
        jk_graphs.clear();
    }

    // Captures the launch sequence of a build just run eagerly (its task tables exist, so the
    // capture allocates nothing) on a private stream of default priority.
    void captureJK(const JKKey &key, const lbx_jk_stats &st)
    {
        if (jk_graphs.size() >= kMaxJKGraphs)
            dropJKGraphs();
        hipStream_t cs = nullptr;
        LBX_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
        hipStream_t saved = stream;
        JKGraph g;
        g.stats = st;
        capturing = true;
        try
        {
            stream = cs;
            LBX_HIP(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
            try
            {
                queueJK(std::get<0>(key), std::get<1>(key), std::get<2>(key), std::get<3>(key), std::get<4>(key),
                        std::get<5>(key) != 0, false);
            }
            catch (...)
            {
                hipGraph_t tmp = nullptr;
                (void)hipStreamEndCapture(cs, &tmp);
                if (tmp)
                    (void)hipGraphDestroy(tmp);
                throw;
            }
            LBX_HIP(hipStreamEndCapture(cs, &g.graph));
            capturing = false;
            stream = saved;
            LBX_HIP(hipGraphInstantiate(&g.exec, g.graph, nullptr, nullptr, 0));
        }
        catch (...)
        {
            capturing = false;
            stream = saved;
            if (g.graph)
                (void)hipGraphDestroy(g.graph);
            (void)hipStreamDestroy(cs);
            throw;
        }
        (void)hipStreamDestroy(cs);
        jk_graphs.emplace(key, g);
    }

    // per-class timing (lbx_profile_enable)
    struct Prof
    {
        lbx_class_profile rec{};
        hipEvent_t start = nullptr, stop = nullptr;
        bool pending = false;
    };
    bool profiling = false;
    std::map<std::tuple<int, int, int>, Prof> prof;   // (bra class, ket class, tier 0 FP64 / 1 FP32)

    ~lbx_context()
    {
        dropRiGraph();
        dropJKGraphs();
        for (auto &kv : prof)
        {
            if (kv.second.start)
                (void)hipEventDestroy(kv.second.start);
            if (kv.second.stop)
                (void)hipEventDestroy(kv.second.stop);
        }
    }

    void collectProfile()
    {
        for (auto &kv : prof)
        {
            Prof &p = kv.second;
            if (!p.pending)
                continue;
            float ms = 0;
            LBX_HIP(hipEventElapsedTime(&ms, p.start, p.stop));
            p.rec.ms += ms;
            p.pending = false;
        }
    }
};

namespace
{
    // A call on a context: one that runs out of device memory frees what the context holds to save
    // time only, and is made again without it.
    template <class F>
    int guardedIn(lbx_context *ctx, F &&f)
    {
        const int rc = guarded(f);
        if (rc != LBX_ERR_NOMEM || !ctx)
            return rc;
        bool freed = false;
        (void)guarded([&] {
            std::lock_guard<std::mutex> lk(ctx->mu);
            (void)hipGetLastError();   // not the next launch's error
            freed = ctx->freeExtras();
            ctx->no_extras = ctx->no_extras || freed;
        });
        return freed ? guarded(f) : rc;
    }

    // Shells, pair classes, E matrices and per-pair molecule ids of a new context.
    void setupContext(lbx_context &ctx, const lbx_basis &main_basis, const lbx_basis *aux_basis)
    {
        Context &c = ctx;
        LBX_HIP(hipGetDevice(&c.device));
        ctx.d_scratch = scratchAddress(c.device);
        c.natoms = main_basis.natoms;
        c.shells = buildShells(main_basis, c.nbf, c.max_l, kMaxLMain);
        if (c.shells.empty())
            throw Error(LBX_ERR_INVALID, "lbx_create: empty main basis");
        if (aux_basis)
        {
            if (aux_basis->natoms != c.natoms)
                throw Error(LBX_ERR_INVALID, "lbx_create: aux basis natoms differs");
            c.shells_aux = buildShells(*aux_basis, c.nbf_aux, c.max_l_aux, kMaxLAux);
        }
        c.d_boys = const_cast<double *>(boysTableDevice());
        buildPairClasses(c);
        for (auto &pc : c.cls)
        {
            computeEcoeffs(c, pc, c.shells);
            pc.d_mol = c.upload(pc.mol);
        }
        for (auto &pc : c.aux)
        {
            computeEcoeffs(c, pc, c.shells_aux);
            pc.d_mol = c.upload(pc.mol);
        }
        LBX_HIP(hipStreamSynchronize(c.stream));
    }

    // Concatenation of several molecules' lbx_basis arrays (atom indices offset).
    struct FlatBatch
    {
        std::vector<double> coords, exps, coeffs;
        std::vector<int> atom, l, nprim;
        int natoms = 0;
        lbx_basis b{};

        void add(const lbx_basis &x)
        {
            if (x.natoms < 0 || x.nshells < 0 || (x.natoms > 0 && !x.coords) ||
                (x.nshells > 0 && (!x.shell_atom || !x.shell_l || !x.shell_nprim || !x.exps || !x.coeffs)))
                throw Error(LBX_ERR_INVALID, "lbx_create_batch: bad basis");
            coords.insert(coords.end(), x.coords, x.coords + 3 * x.natoms);
            long long np = 0;
            for (int s = 0; s < x.nshells; s++)
            {
                if (x.shell_atom[s] < 0 || x.shell_atom[s] >= x.natoms || x.shell_nprim[s] <= 0)
                    throw Error(LBX_ERR_INVALID, "lbx_create_batch: bad shell");
                atom.push_back(x.shell_atom[s] + natoms);
                l.push_back(x.shell_l[s]);
                nprim.push_back(x.shell_nprim[s]);
                np += x.shell_nprim[s];
            }
            exps.insert(exps.end(), x.exps, x.exps + np);
            coeffs.insert(coeffs.end(), x.coeffs, x.coeffs + np);
            natoms += x.natoms;
        }

        const lbx_basis &view()
        {
            b = lbx_basis{natoms, coords.data(), static_cast<int>(l.size()), atom.data(), l.data(),
                          nprim.data(), exps.data(), coeffs.data()};
            return b;
        }
    };
}

extern "C"
{
    const char *lbx_last_error(void) { return g_err.c_str(); }

    int lbx_create(lbx_context **out, const lbx_basis *main_basis, const lbx_basis *aux_basis)
    {
        if (!out || !main_basis)
        {
            g_err = "lbx_create: null argument";
            return LBX_ERR_INVALID;
        }
        *out = nullptr;
        auto ctx = std::make_unique<lbx_context>();
        int rc = guarded([&] { setupContext(*ctx, *main_basis, aux_basis); });
        if (rc != LBX_OK)
        {
            ctx->release();
            return rc;
        }
        *out = ctx.release();
        return LBX_OK;
    }

    int lbx_create_batch(lbx_context **out, int nmol, const lbx_basis *main_bases,
                         const lbx_basis *aux_bases)
    {
        if (!out || !main_bases || !aux_bases || nmol <= 0)
        {
            g_err = "lbx_create_batch: null argument or nmol <= 0";
            return LBX_ERR_INVALID;
        }
        *out = nullptr;
        auto ctx = std::make_unique<lbx_context>();
        int rc = guarded([&]
                         {
                             // one basis over all molecules' atoms, atoms grouped by molecule
                             FlatBatch m, a;
                             for (int k = 0; k < nmol; k++)
                             {
                                 if (main_bases[k].natoms != aux_bases[k].natoms)
                                     throw Error(LBX_ERR_INVALID, "lbx_create_batch: aux basis natoms differs");
                                 for (int i = 0; i < main_bases[k].natoms; i++)
                                     ctx->atom_mol.push_back(k);
                                 m.add(main_bases[k]);
                                 a.add(aux_bases[k]);
                             }
                             ctx->nmol = nmol;
                             setupContext(*ctx, m.view(), &a.view());
                         });
        if (rc != LBX_OK)
        {
            ctx->release();
            return rc;
        }
        *out = ctx.release();
        return LBX_OK;
    }

    int lbx_destroy(lbx_context *ctx)
    {
        if (!ctx)
            return LBX_OK;
        int rc = guarded([&]
                         {
                             (void)hipStreamSynchronize(ctx->stream);
                             ctx->release();
                         });
        delete ctx;
        return rc;
    }

    int lbx_dims(const lbx_context *ctx, long *nbf, long *nbf_aux, long *natoms)
    {
        if (!ctx)
        {
            g_err = "lbx_dims: null context";
            return LBX_ERR_INVALID;
        }
        if (nbf)
            *nbf = static_cast<long>(ctx->nbf);
        if (nbf_aux)
            *nbf_aux = static_cast<long>(ctx->nbf_aux);
        if (natoms)
            *natoms = ctx->natoms;
        return LBX_OK;
    }

    int lbx_set_stream(lbx_context *ctx, void *stream)
    {
        if (!ctx)
        {
            g_err = "lbx_set_stream: null context";
            return LBX_ERR_INVALID;
        }
        ctx->stream = static_cast<hipStream_t>(stream);
        return LBX_OK;
    }

    int lbx_set_memory_limit(lbx_context *ctx, long bytes)
    {
        return guarded([&]
                       {
                           if (!ctx || bytes < 0)
                               throw Error(LBX_ERR_INVALID, "lbx_set_memory_limit: null context or negative limit");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           bool over = false;
                           {
                               std::lock_guard<std::mutex> la(ctx->alloc_mu);
                               ctx->limit = static_cast<size_t>(bytes);
                               over = bytes > 0 && ctx->held > ctx->limit;
                           }
                           ctx->no_extras = false;
                           if (over)
                               ctx->freeExtras();
                           // sums prepared without the copies would stay so
                           ctx->dropRiGraph();
                           ctx->ri_prepared.clear();
                       });
    }

    int lbx_synchronize(lbx_context *ctx)
    {
        if (!ctx)
        {
            g_err = "lbx_synchronize: null context";
            return LBX_ERR_INVALID;
        }
        return guarded([&] { LBX_HIP(hipStreamSynchronize(ctx->stream)); });
    }

    int lbx_boys(int n, long count, const double *x, double *out, void *stream)
    {
        return guarded([&]
                       {
                           if (n < 0 || n > kMaxLBoys || count < 0 || (count > 0 && (!x || !out)))
                               throw Error(LBX_ERR_INVALID, "lbx_boys: bad argument");
                           if (count == 0)
                               return;
                           static const auto fns = boysFns(std::make_integer_sequence<int, kMaxLBoys + 1>{});
                           fns[n](count, x, out, boysTableDevice(), static_cast<hipStream_t>(stream));
                           LBX_HIP(hipGetLastError());
                       });
    }

    int lbx_eri4(lbx_context *ctx, double *out)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !out)
                               throw Error(LBX_ERR_INVALID, "lbx_eri4: null argument");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           Context &c = *ctx;
                           requireSingle(c, "lbx_eri4");
                           const long long n = static_cast<long long>(c.nbf);
                           if (!allPairs(c))
                               fill(out, n * n * n * n, 0.0, c.stream);
                           KArgs extra{};
                           extra.out = out;
                           extra.kind = 4;
                           std::vector<PlainJob> jobs;
                           for (size_t i = 0; i < c.cls.size(); i++)
                               for (size_t j = 0; j <= i; j++)
                                   jobs.push_back({MODE_DENSE, &c.cls[i], &c.cls[j], Pairing::Unique, i == j, extra});
                           ctx->runPlain(jobs);
                       });
    }

    int lbx_eri4_diag(lbx_context *ctx, double *out)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !out)
                               throw Error(LBX_ERR_INVALID, "lbx_eri4_diag: null argument");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           Context &c = *ctx;
                           requireSingle(c, "lbx_eri4_diag");
                           const long long n = static_cast<long long>(c.nbf);
                           fill(out, n * n, 0.0, c.stream);
                           size_t pairs = 0;
                           for (auto &pc : c.cls)
                               pairs += pc.n_pairs;
                           DevBuf q(pairs);
                           std::vector<PlainJob> jobs;
                           pairs = 0;
                           for (auto &pc : c.cls)
                           {
                               KArgs extra{};
                               extra.qout = q.p + pairs;
                               extra.dout = out;
                               extra.kind = 4;
                               jobs.push_back({MODE_DIAG, &pc, &pc, Pairing::Diagonal, true, extra});
                               pairs += pc.n_pairs;
                           }
                           ctx->runPlain(jobs);
                       });
    }

    int lbx_eri3(lbx_context *ctx, double *out)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !out)
                               throw Error(LBX_ERR_INVALID, "lbx_eri3: null argument");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           Context &c = *ctx;
                           requireSingle(c, "lbx_eri3");
                           if (c.shells_aux.empty())
                               throw Error(LBX_ERR_STATE, "eri3(): RI approximation is not enabled");
                           const long long n = static_cast<long long>(c.nbf);
                           if (!allPairs(c))
                               fill(out, n * n * static_cast<long long>(c.nbf_aux), 0.0, c.stream);
                           KArgs extra{};
                           extra.out = out;
                           extra.kind = 3;
                           std::vector<PlainJob> jobs;
                           for (auto &bra : c.cls)
                               for (auto &ket : c.aux)
                                   jobs.push_back({MODE_DENSE, &bra, &ket, Pairing::All, false, extra});
                           ctx->runPlain(jobs);
                       });
    }

    int lbx_eri2(lbx_context *ctx, double *out)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !out)
                               throw Error(LBX_ERR_INVALID, "lbx_eri2: null argument");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           Context &c = *ctx;
                           requireSingle(c, "lbx_eri2");
                           if (c.shells_aux.empty())
                               throw Error(LBX_ERR_STATE, "eri2(): RI approximation is not enabled");
                           const long long n = static_cast<long long>(c.nbf_aux);
                           fill(out, n * n, 0.0, c.stream);
                           KArgs extra{};
                           extra.out = out;
                           extra.kind = 2;
                           std::vector<PlainJob> jobs;
                           for (size_t i = 0; i < c.aux.size(); i++)
                               for (size_t j = 0; j <= i; j++)
                                   jobs.push_back({MODE_DENSE, &c.aux[i], &c.aux[j], Pairing::Unique, i == j, extra});
                           ctx->runPlain(jobs);
                       });
    }

    int lbx_eri2_diag(lbx_context *ctx, double *out)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !out)
                               throw Error(LBX_ERR_INVALID, "lbx_eri2_diag: null argument");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           Context &c = *ctx;
                           requireSingle(c, "lbx_eri2_diag");
                           if (c.shells_aux.empty())
                               throw Error(LBX_ERR_STATE, "eri2Diagonal(): RI approximation is not enabled");
                           fill(out, static_cast<long long>(c.nbf_aux), 0.0, c.stream);
                           size_t pairs = 0;
                           for (auto &pc : c.aux)
                               pairs += pc.n_pairs;
                           DevBuf q(pairs);
                           std::vector<PlainJob> jobs;
                           pairs = 0;
                           for (auto &pc : c.aux)
                           {
                               KArgs extra{};
                               extra.qout = q.p + pairs;
                               extra.dout = out;
                               extra.kind = 2;
                               jobs.push_back({MODE_DIAG, &pc, &pc, Pairing::Diagonal, true, extra});
                               pairs += pc.n_pairs;
                           }
                           ctx->runPlain(jobs);
                       });
    }

    // Dense derivative tensors (kind 4, 3, 2): every unique class pair's unique quartets, one
    // launch per class pair, each writing its blocks' images.
    namespace
    {
        void runD1(Context &c, int kind, double *out)
        {
            const long long n = static_cast<long long>(c.nbf), nx = static_cast<long long>(c.nbf_aux);
            const long long total = kind == 4 ? 12 * n * n * n * n : (kind == 3 ? 9 * n * n * nx : 6 * nx * nx);
            fill(out, total, 0.0, c.stream);
            if (kind != 2)
                for (auto &pc : c.cls)
                    computeEcoeffsD1(c, pc);
            std::vector<void *> bufs;
            auto one = [&](const PairClass &bra, const PairClass &ket, bool same)
            {
                if (bra.n_pairs == 0 || ket.n_pairs == 0)
                    return;
                std::vector<int> tasks;
                for (int p = 0; p < bra.n_pairs; p++)
                    for (int q = 0; q < (same ? p + 1 : ket.n_pairs); q++)
                    {
                        tasks.push_back(p);
                        tasks.push_back(q);
                    }
                void *d = nullptr;
                LBX_HIP(hipMalloc(&d, tasks.size() * sizeof(int)));
                bufs.push_back(d);
                LBX_HIP(hipMemcpyAsync(d, tasks.data(), tasks.size() * sizeof(int), hipMemcpyHostToDevice,
                                       c.stream));
                D1Args a{};
                a.bra = bra.view();
                a.ket = ket.view();
                a.la = bra.la;
                a.lb = bra.lb;
                a.lc = ket.la;
                a.ld = ket.lb;
                a.bra_single = bra.single ? 1 : 0;
                a.ket_single = ket.single ? 1 : 0;
                a.tasks = static_cast<const int *>(d);
                a.ntasks = static_cast<long long>(tasks.size() / 2);
                a.boys = c.d_boys;
                a.out = out;
                a.kind = kind;
                a.nbf = n;
                a.naux = nx;
                launchD1(a, c.stream);
                // the host task list must outlive the asynchronous copy
                LBX_HIP(hipStreamSynchronize(c.stream));
            };
            try
            {
                if (kind == 4)
                {
                    for (size_t i = 0; i < c.cls.size(); i++)
                        for (size_t j = 0; j <= i; j++)
                            one(c.cls[i], c.cls[j], i == j);
                }
                else if (kind == 3)
                {
                    for (auto &bra : c.cls)
                        for (auto &ket : c.aux)
                            one(bra, ket, false);
                }
                else
                {
                    for (size_t i = 0; i < c.aux.size(); i++)
                        for (size_t j = 0; j <= i; j++)
                            one(c.aux[i], c.aux[j], i == j);
                }
            }
            catch (...)
            {
                (void)hipStreamSynchronize(c.stream);
                for (void *d : bufs)
                    (void)hipFree(d);
                throw;
            }
            LBX_HIP(hipStreamSynchronize(c.stream));
            for (void *d : bufs)
                (void)hipFree(d);
        }
    }

    // Blocks of listed shell quartets / triplets / doublets (kind 4, 3, 2) in the caller's
    // shell order: the integrals themselves, their first derivatives, the spin-orbit-type
    // integrals (kinds 4, 3) or the second derivatives (kind 2) (op: D1_OP_*); every entry of
    // one call has the same angular momenta.  Entries whose shell pair has no primitive pair
    // above the 1e-15 screen (the reference's ShellPairData drops such pairs) are zero.
    namespace
    {
        // (shell a, shell b) of a pair class -> pair index, made on first use
        const std::unordered_map<long long, int> &pairIndex(Context &c, std::vector<std::unordered_map<long long, int>> &maps,
                                                           int cls_idx)
        {
            if (maps.size() < c.cls.size())
                maps.resize(c.cls.size());
            auto &m = maps[cls_idx];
            const PairClass &pc = c.cls[cls_idx];
            if (m.empty() && pc.n_pairs > 0)
            {
                const long long nsh = static_cast<long long>(c.shells.size());
                for (int p = 0; p < pc.n_pairs; p++)
                    m.emplace(static_cast<long long>(pc.sh_a[p]) * nsh + pc.sh_b[p], p);
            }
            return m;
        }

        void runBlocks(lbx_context &c, std::vector<std::unordered_map<long long, int>> &maps, int kind,
                       int op, long long nq, const int *sh, double *out, const char *who,
                       int *staging = nullptr)
        {
            const int per = kind == 4 ? 4 : (kind == 3 ? 3 : 2);
            const int nsh = static_cast<int>(c.shells.size()), nax = static_cast<int>(c.shells_aux.size());
            auto isAux = [&](int pos) { return kind == 2 || (kind == 3 && pos == 2); };
            auto lOf = [&](int pos, int idx) {
                const int n = isAux(pos) ? nax : nsh;
                if (idx < 0 || idx >= n)
                    throw Error(LBX_ERR_INVALID, std::string(who) + ": shell index " + std::to_string(idx) +
                                                         " out of range");
                return isAux(pos) ? c.shells_aux[idx].l : c.shells[idx].l;
            };
            if (nq == 0)
                return;
            int l[4] = {0, 0, 0, 0};
            for (int k = 0; k < per; k++)
                l[k] = lOf(k, sh[k]);
            for (long long t = 0; t < nq; t++)
                for (int k = 0; k < per; k++)
                    if (lOf(k, sh[per * t + k]) != l[k])
                        throw Error(LBX_ERR_INVALID, std::string(who) + ": every entry must have the "
                                                                        "angular momenta of the first");
            const int ncomp = op == D1_OP_PLAIN ? 1 : op == D1_OP_SOC ? 3 : op == D1_OP_D2 ? 36
                                                                                       : 3 * (kind == 4 ? 4 : (kind == 3 ? 3 : 2));
            long long bsize = 1;
            for (int k = 0; k < per; k++)
                bsize *= nSph(l[k]);
            // library pair classes of the two sides
            PairClass *bra, *ket;
            int ibra = -1, iket = -1;
            if (kind == 2)
            {
                bra = &c.aux[l[0]];
                ket = &c.aux[l[1]];
            }
            else
            {
                ibra = pairClassIdx(std::max(l[0], l[1]), std::min(l[0], l[1]));
                bra = &c.cls[ibra];
                if (kind == 4)
                {
                    iket = pairClassIdx(std::max(l[2], l[3]), std::min(l[2], l[3]));
                    ket = &c.cls[iket];
                }
                else
                    ket = &c.aux[l[2]];
            }
            // pair of two main shells in the library's order (l_a > l_b, or equal l and a >= b)
            auto mainPair = [&](int cls_idx, int a, int b, bool &swapped) {
                swapped = c.shells[a].l < c.shells[b].l || (c.shells[a].l == c.shells[b].l && a < b);
                const long long key = static_cast<long long>(swapped ? b : a) * nsh + (swapped ? a : b);
                const auto &m = pairIndex(c, maps, cls_idx);
                auto it = m.find(key);
                return it == m.end() ? -1 : it->second;
            };
            // single auxiliary shell -> its position in the class of its l
            auto auxPair = [&](const PairClass &pc, int s) {
                auto it = std::lower_bound(pc.sh_a.begin(), pc.sh_a.end(), s);
                return it != pc.sh_a.end() && *it == s ? static_cast<int>(it - pc.sh_a.begin()) : -1;
            };
            // The integrals themselves: the compiled one-wave kernel of the class pair, whose bra is
            // the side with the higher class (or higher l of two auxiliary shells); the run-time-L
            // kernel for derivatives and for the class pairs with a main g shell that it does not cover
            // (it covers (gs|ls): the instances of auxiliary g shells).
            const bool flip = kind == 2 ? bra->la < ket->la
                                        : kernelSlot(MODE_BLOCK, bra->la, bra->lb, ket->la, ket->lb, VAR_MFMA).fn == nullptr;
            const KernelSlot *wave = nullptr;
            if (op == D1_OP_PLAIN)
                wave = flip ? &kernelSlot(MODE_BLOCK, ket->la, ket->lb, bra->la, bra->lb, VAR_MFMA)
                            : &kernelSlot(MODE_BLOCK, bra->la, bra->lb, ket->la, ket->lb, VAR_MFMA);
            if (wave && !wave->fn)
                wave = nullptr;
            std::vector<int> tasks;
            tasks.reserve(4 * nq);
            for (long long t = 0; t < nq; t++)
            {
                const int *e = sh + per * t;
                bool sab = false, scd = false;
                int p, q;
                if (kind == 2)
                {
                    p = auxPair(*bra, e[0]);
                    q = auxPair(*ket, e[1]);
                }
                else
                {
                    p = mainPair(ibra, e[0], e[1], sab);
                    q = kind == 4 ? mainPair(iket, e[2], e[3], scd) : auxPair(*ket, e[2]);
                }
                if (p < 0 || q < 0)
                    continue;
                if (wave && flip)
                    tasks.insert(tasks.end(), {q, p, (scd ? 1 : 0) | (sab ? 2 : 0) | 4, static_cast<int>(t)});
                else
                    tasks.insert(tasks.end(), {p, q, (sab ? 1 : 0) | (scd ? 2 : 0), static_cast<int>(t)});
            }
            // entries without a task stay zero; the one-wave kernel writes every element of the others
            if (!wave || static_cast<long long>(tasks.size()) < 4 * nq)
                fill(out, nq * ncomp * bsize, 0.0, c.stream);
            if (tasks.empty())
                return;
            if (op == D1_OP_DERIV || op == D1_OP_SOC)
            {
                if (kind != 2)
                    computeEcoeffsD1(c, *bra);
                if (kind == 4 && op == D1_OP_DERIV)
                    computeEcoeffsD1(c, *ket);
            }
            // the task list: in the device's scratch array (staging != nullptr: the allocation-free
            // entry, at most kStaticEntries entries), in the context's buffer (lists of up to
            // kBlockTaskInts ints), or in a buffer of this call
            const bool kept = !staging && tasks.size() <= lbx_context::kBlockTaskInts;
            void *d = staging;
            if (kept)
            {
                if (!c.block_tasks)
                    c.block_tasks = c.alloc<int>(lbx_context::kBlockTaskInts);
                d = c.block_tasks;
            }
            else if (!staging)
                LBX_HIP(hipMalloc(&d, tasks.size() * sizeof(int)));
            try
            {
                LBX_HIP(hipMemcpyAsync(d, tasks.data(), tasks.size() * sizeof(int), hipMemcpyHostToDevice,
                                       c.stream));
                if (wave)
                {
                    KArgs a{};
                    a.bra = (flip ? ket : bra)->view();
                    a.ket = (flip ? bra : ket)->view();
                    a.plo = static_cast<const int *>(d);
                    a.ntasks = static_cast<long long>(tasks.size() / 4);
                    a.boys = c.d_boys;
                    a.out = out;
                    wave->fn(a, c.stream);
                    LBX_HIP(hipGetLastError());
                }
                else
                {
                    D1Args a{};
                    a.bra = bra->view();
                    a.ket = ket->view();
                    a.la = bra->la;
                    a.lb = bra->lb;
                    a.lc = ket->la;
                    a.ld = ket->lb;
                    a.bra_single = bra->single ? 1 : 0;
                    a.ket_single = ket->single ? 1 : 0;
                    a.tasks = static_cast<const int *>(d);
                    a.ntasks = static_cast<long long>(tasks.size() / 4);
                    a.boys = c.d_boys;
                    a.out = out;
                    a.kind = kind;
                    a.nbf = static_cast<long long>(c.nbf);
                    a.naux = static_cast<long long>(c.nbf_aux);
                    a.blocks = 1;
                    a.op = op;
                    launchD1(a, c.stream);
                }
                LBX_HIP(hipStreamSynchronize(c.stream));
            }
            catch (...)
            {
                (void)hipStreamSynchronize(c.stream);
                if (!staging && !kept)
                    (void)hipFree(d);
                throw;
            }
            if (!staging && !kept)
                (void)hipFree(d);
        }

        int blocksEntry(lbx_context *ctx, int kind, int op, long nq, const int *shells, double *out,
                        const char *who, bool no_alloc = false)
        {
            return guardedIn(ctx, [&]
                           {
                               if (!ctx || nq < 0 || (nq > 0 && (!shells || !out)))
                                   throw Error(LBX_ERR_INVALID, std::string(who) + ": null argument or negative count");
                               if (no_alloc && nq > kStaticEntries)
                                   throw Error(LBX_ERR_INVALID, std::string(who) + ": " + std::to_string(nq) +
                                                                        " entries, at most " +
                                                                        std::to_string(kStaticEntries) + " per call");
                               std::lock_guard<std::mutex> lk(ctx->mu);
                               requireSingle(*ctx, who);
                               if (kind != 4 && ctx->shells_aux.empty())
                                   throw Error(LBX_ERR_STATE, std::string(who) + ": RI approximation is not enabled");
                               runBlocks(*ctx, ctx->pair_maps, kind, op, nq, shells, out, who,
                                         no_alloc ? ctx->d_scratch : nullptr);
                           });
        }
    }

    int lbx_eri4_batch_static(lbx_context *ctx, long nq, const int *shells, double *out)
    {
        return blocksEntry(ctx, 4, D1_OP_PLAIN, nq, shells, out, "lbx_eri4_batch_static", true);
    }

    int lbx_eri4_batch(lbx_context *ctx, long nq, const int *shells, double *out)
    {
        return blocksEntry(ctx, 4, D1_OP_PLAIN, nq, shells, out, "lbx_eri4_batch");
    }

    int lbx_eri3_batch(lbx_context *ctx, long nq, const int *shells, double *out)
    {
        return blocksEntry(ctx, 3, D1_OP_PLAIN, nq, shells, out, "lbx_eri3_batch");
    }

    int lbx_eri2_batch(lbx_context *ctx, long nq, const int *shells, double *out)
    {
        return blocksEntry(ctx, 2, D1_OP_PLAIN, nq, shells, out, "lbx_eri2_batch");
    }

    int lbx_eri4d1_batch(lbx_context *ctx, long nq, const int *shells, double *out)
    {
        return blocksEntry(ctx, 4, D1_OP_DERIV, nq, shells, out, "lbx_eri4d1_batch");
    }

    int lbx_eri3d1_batch(lbx_context *ctx, long nq, const int *shells, double *out)
    {
        return blocksEntry(ctx, 3, D1_OP_DERIV, nq, shells, out, "lbx_eri3d1_batch");
    }

    int lbx_eri2d1_batch(lbx_context *ctx, long nq, const int *shells, double *out)
    {
        return blocksEntry(ctx, 2, D1_OP_DERIV, nq, shells, out, "lbx_eri2d1_batch");
    }

    int lbx_eri4soc_batch(lbx_context *ctx, long nq, const int *shells, double *out)
    {
        return blocksEntry(ctx, 4, D1_OP_SOC, nq, shells, out, "lbx_eri4soc_batch");
    }

    int lbx_eri3soc_batch(lbx_context *ctx, long nq, const int *shells, double *out)
    {
        return blocksEntry(ctx, 3, D1_OP_SOC, nq, shells, out, "lbx_eri3soc_batch");
    }

    int lbx_eri2d2_batch(lbx_context *ctx, long nq, const int *shells, double *out)
    {
        return blocksEntry(ctx, 2, D1_OP_D2, nq, shells, out, "lbx_eri2d2_batch");
    }

    int lbx_eri4d1(lbx_context *ctx, double *out)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !out)
                               throw Error(LBX_ERR_INVALID, "lbx_eri4d1: null argument");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           requireSingle(*ctx, "lbx_eri4d1");
                           runD1(*ctx, 4, out);
                       });
    }

    int lbx_eri3d1(lbx_context *ctx, double *out)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !out)
                               throw Error(LBX_ERR_INVALID, "lbx_eri3d1: null argument");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           requireSingle(*ctx, "lbx_eri3d1");
                           if (ctx->shells_aux.empty())
                               throw Error(LBX_ERR_STATE, "eri3d1: RI approximation is not enabled");
                           runD1(*ctx, 3, out);
                       });
    }

    int lbx_eri2d1(lbx_context *ctx, double *out)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !out)
                               throw Error(LBX_ERR_INVALID, "lbx_eri2d1: null argument");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           requireSingle(*ctx, "lbx_eri2d1");
                           if (ctx->shells_aux.empty())
                               throw Error(LBX_ERR_STATE, "eri2d1: RI approximation is not enabled");
                           runD1(*ctx, 2, out);
                       });
    }

    lbx_jk_stats lbx_context::queueJK(const double *D, double *J, double *K, double schwarz_thresh,
                                      double split, bool mixed, bool prof_on)
    {
        Context &c = *this;
        const long long n = static_cast<long long>(c.nbf);
        fill(J, n * n, 0.0, c.stream);
        fill(K, n * n, 0.0, c.stream);
        // J in parts: launch (i, j) adds to part (i + j) mod the number of classes, so the
        // contributions to a pair's J from each class meet in a part of their own.  An addition
        // rounds to the running sum's last place, and the one-wave forms make one per quartet:
        // in one sum, differences of J builds at 60 atoms (1800 functions) carry 1e-16 of the
        // energy of noise, ten times that of forms which add 64 quartets at once.  Small systems,
        // whose sums are short, and parts of more than 4 GiB go without.
        const int ncls = static_cast<int>(c.cls.size());
        int nparts = n < 400 ? 1 : static_cast<int>(std::clamp<long long>((4LL << 30) / (8 * n * n), 1, ncls));
        if (nparts > 1 && !j_parts)
            j_parts = takeExtra<double>((nparts - 1) * n * n);
        if (!j_parts)
            nparts = 1;
        if (nparts > 1)
            fill(j_parts, (nparts - 1) * n * n, 0.0, c.stream);
        lbx_jk_stats st{};
        std::vector<QueuedLaunch> queue;
        auto launch = [&](int i, int j, int tier, int var, double lo, double hi)
        {
            const PairClass &bra = c.cls[i], &ket = c.cls[j];
            const int part = (i + j) % nparts;
            const JKLaunch l = prepareJK(i, j, var, D, part ? j_parts + (part - 1) * n * n : J, K, lo, hi);
            const TaskTable &t = *l.t;
            var = l.var;
            st.quartets += t.quartets;
            st.flops += t.flops;
            if (isF32Variant(var))
                st.quartets_fp32 += t.quartets;
            if (!prof_on)
            {
                const KernelSlot &slot = kernelSlot(MODE_JK, bra.la, bra.lb, ket.la, ket.lb, var);
                queue.push_back({l.fn, l.a, variantTime(MODE_JK, bra, ket, slot, isF32Variant(var), t.quartets, t.quartets / 64)});
                return;
            }
            // one class pair at a time on the context stream, an event pair around each
            Prof &pr = prof[{i, j, tier}];
            if (!pr.start)
            {
                LBX_HIP(hipEventCreate(&pr.start));
                LBX_HIP(hipEventCreate(&pr.stop));
                pr.rec.la = bra.la;
                pr.rec.lb = bra.lb;
                pr.rec.lc = ket.la;
                pr.rec.ld = ket.lb;
            }
            pr.rec.kernel = var;
            flushStaged();
            LBX_HIP(hipEventRecord(pr.start, c.stream));
            l.fn(l.a, c.stream);
            LBX_HIP(hipGetLastError());
            LBX_HIP(hipEventRecord(pr.stop, c.stream));
            pr.pending = true;
            pr.rec.calls += 1;
            pr.rec.quartets += t.quartets;
            pr.rec.flops += t.flops;
        };
        for (int i = 0; i < static_cast<int>(c.cls.size()); i++)
            for (int j = 0; j <= i; j++)
            {
                if (c.cls[i].n_pairs == 0 || c.cls[j].n_pairs == 0)
                    continue;
                if (filter_i >= 0 && (i != filter_i || j != filter_j))
                    continue;
                // the tiers [split, inf) and [schwarz, split), cut to the bound window
                const double lo0 = std::max(split, window_lo), hi0 = window_hi;
                const double lo1 = std::max(schwarz_thresh, window_lo), hi1 = std::min(split, window_hi);
                if (lo0 < hi0)
                    launch(i, j, 0, variantFor(i, j, lo0, hi0), lo0, hi0);
                if (mixed && lo1 < hi1)
                    launch(i, j, 1, variant32For(i, j, lo1, hi1), lo1, hi1);
            }
        flushStaged();
        Fan fan(side, c.stream, queue.size() > 1);
        launchAll(queue, fan);
        const int gridn = static_cast<int>(std::min<long long>((n * n + 255) / 256, 65536));
        hipLaunchKernelGGL(symmetrizeKernel, dim3(gridn), dim3(256), 0, c.stream, J, static_cast<int>(n), j_parts,
                           nparts - 1);
        hipLaunchKernelGGL(symmetrizeKernel, dim3(gridn), dim3(256), 0, c.stream, K, static_cast<int>(n),
                           nullptr, 0);
        LBX_HIP(hipGetLastError());
        return st;
    }

    int lbx_jk(lbx_context *ctx, const double *D, double *J, double *K, double schwarz_thresh,
               int precision, double mixed_thresh, lbx_jk_stats *stats)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !D || !J || !K)
                               throw Error(LBX_ERR_INVALID, "lbx_jk: null argument");
                           if (precision != LBX_FP64 && precision != LBX_MIXED)
                               throw Error(LBX_ERR_INVALID, "lbx_jk: precision must be LBX_FP64 or LBX_MIXED");
                           if (!(schwarz_thresh >= 0))
                               throw Error(LBX_ERR_INVALID, "lbx_jk: negative Schwarz threshold");
                           if (precision == LBX_MIXED && !(mixed_thresh >= 0))
                               throw Error(LBX_ERR_INVALID, "lbx_jk: negative mixed-precision threshold");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           Context &c = *ctx;
                           requireSingle(c, "lbx_jk");
                           ctx->ensureSchwarz();
                           // quartets with schwarz <= Q_ab Q_cd < split run in FP32
                           const bool mixed = precision == LBX_MIXED && mixed_thresh > schwarz_thresh;
                           const double split = mixed ? mixed_thresh : schwarz_thresh;
                           if (mixed)
                               ensureF32(c);
                           // Replays: the launch sequence of a (D, J, K, thresholds) set is
                           // captured into a HIP graph after its first (eager) build and replayed
                           // on later calls; per-class timing and the class filter run eagerly.
                           const bool graphs = ctx->graphs && !ctx->profiling && ctx->filter_i < 0 &&
                                               ctx->window_lo <= 0.0 && ctx->window_hi == kNoUpper;
                           const lbx_context::JKKey gkey{D, J, K, schwarz_thresh, split, mixed ? 1 : 0};
                           if (graphs)
                           {
                               auto it = ctx->jk_graphs.find(gkey);
                               if (it != ctx->jk_graphs.end())
                               {
                                   LBX_HIP(hipGraphLaunch(it->second.exec, c.stream));
                                   LBX_HIP(hipStreamSynchronize(c.stream));
                                   if (stats)
                                       *stats = it->second.stats;
                                   return;
                               }
                           }
                           lbx_jk_stats st = ctx->queueJK(D, J, K, schwarz_thresh, split, mixed, ctx->profiling);
                           LBX_HIP(hipStreamSynchronize(c.stream));
                           if (ctx->profiling)
                               ctx->collectProfile();
                           if (graphs)
                               ctx->captureJK(gkey, st);
                           if (stats)
                               *stats = st;
                       });
    }

    int lbx_ri_sums(lbx_context *ctx, double *out, int precision, double mixed_thresh,
                    lbx_ri_stats *stats)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !out)
                               throw Error(LBX_ERR_INVALID, "lbx_ri_sums: null argument");
                           if (precision != LBX_FP64 && precision != LBX_MIXED)
                               throw Error(LBX_ERR_INVALID, "lbx_ri_sums: precision must be LBX_FP64 or LBX_MIXED");
                           if (precision == LBX_MIXED && !(mixed_thresh >= 0))
                               throw Error(LBX_ERR_INVALID, "lbx_ri_sums: negative mixed-precision threshold");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           Context &c = *ctx;
                           if (c.shells_aux.empty())
                               throw Error(LBX_ERR_STATE, "lbx_ri_sums: the context has no auxiliary basis");
                           const double split = precision == LBX_MIXED ? mixed_thresh : 0.0;
                           auto report = [&]
                           {
                               if (stats)
                               {
                                   stats->triplets = ctx->ri_triplets;
                                   stats->doublets = ctx->ri_doublets;
                                   stats->flops = ctx->ri_flops;
                                   stats->triplets_fp32 = ctx->ri_triplets32;
                                   stats->doublets_fp32 = ctx->ri_doublets32;
                               }
                           };
                           if (!ctx->graphs)
                           {
                               // eager launches on the context stream
                               if (split > 0.0)
                               {
                                   ctx->ensureSchwarz();
                                   ctx->ensureSchwarzAux();
                                   ensureF32(c);
                                   ensureF32Aux(c);
                               }
                               ctx->prepareRiSums(split);
                               ctx->queueRiSums(out, c.stream);
                               LBX_HIP(hipStreamSynchronize(c.stream));
                               report();
                               return;
                           }
                           if (!ctx->ri_exec || ctx->ri_out != out || ctx->ri_split != split)
                           {
                               ctx->dropRiGraph();
                               if (split > 0.0)
                               {
                                   ctx->ensureSchwarz();
                                   ctx->ensureSchwarzAux();
                                   ensureF32(c);
                                   ensureF32Aux(c);
                               }
                               ctx->prepareRiSums(split);
                               ctx->ri_split = split;
                               // capture on a private stream (default priority), replay on the
                               // context stream
                               hipStream_t cs = nullptr;
                               LBX_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
                               try
                               {
                                   LBX_HIP(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
                                   try
                                   {
                                       ctx->queueRiSums(out, cs);
                                   }
                                   catch (...)
                                   {
                                       hipGraph_t g = nullptr;
                                       (void)hipStreamEndCapture(cs, &g);
                                       if (g)
                                           (void)hipGraphDestroy(g);
                                       throw;
                                   }
                                   LBX_HIP(hipStreamEndCapture(cs, &ctx->ri_graph));
                                   LBX_HIP(hipGraphInstantiate(&ctx->ri_exec, ctx->ri_graph, nullptr, nullptr, 0));
                               }
                               catch (...)
                               {
                                   (void)hipStreamDestroy(cs);
                                   ctx->dropRiGraph();
                                   throw;
                               }
                               (void)hipStreamDestroy(cs);
                               ctx->ri_out = out;
                           }
                           LBX_HIP(hipGraphLaunch(ctx->ri_exec, c.stream));
                           LBX_HIP(hipStreamSynchronize(c.stream));
                           report();
                       });
    }

    int lbx_set_graphs(lbx_context *ctx, int on)
    {
        return guarded([&]
                       {
                           if (!ctx)
                               throw Error(LBX_ERR_INVALID, "lbx_set_graphs: null context");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           ctx->graphs = on != 0;
                           if (!ctx->graphs)
                           {
                               ctx->dropJKGraphs();
                               ctx->dropRiGraph();
                           }
                       });
    }

    int lbx_jk_grad(lbx_context *ctx, const double *D, double *grad, double schwarz_thresh,
                    int precision, double mixed_thresh, lbx_jk_stats *stats)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !D || !grad)
                               throw Error(LBX_ERR_INVALID, "lbx_jk_grad: null argument");
                           if (!(schwarz_thresh >= 0))
                               throw Error(LBX_ERR_INVALID, "lbx_jk_grad: negative Schwarz threshold");
                           if (precision != LBX_FP64 && precision != LBX_MIXED)
                               throw Error(LBX_ERR_INVALID, "lbx_jk_grad: precision must be LBX_FP64 or LBX_MIXED");
                           if (precision == LBX_MIXED && !(mixed_thresh >= 0))
                               throw Error(LBX_ERR_INVALID, "lbx_jk_grad: negative mixed-precision threshold");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           Context &c = *ctx;
                           requireSingle(c, "lbx_jk_grad");
                           ctx->ensureSchwarz();
                           for (auto &pc : c.cls)
                               computeEcoeffsD1(c, pc);
                           const bool mixed = precision == LBX_MIXED && mixed_thresh > schwarz_thresh;
                           if (mixed)
                           {
                               ensureF32(c);
                               ensureF32D1(c);
                           }
                           const long long ng = 3LL * c.natoms;
                           if (!ctx->grad_copies)
                               ctx->grad_copies = c.alloc<double>(lbx_context::kGradCopies * ng);
                           fill(ctx->grad_copies, lbx_context::kGradCopies * ng, 0.0, c.stream);
                           double nq = 0, fl = 0, nq32 = 0;
                           std::vector<std::pair<double, lbx_context::GradLaunch>> queue;
                           auto add = [&](int i, int j, double lo, double hi, bool fp32)
                           {
                               const PairClass &bra = c.cls[i], &ket = c.cls[j];
                               const auto l = ctx->prepareGrad(i, j, D, lo, hi, fp32);
                               const double f = gradFlops(*l.t, bra.la, bra.lb, ket.la, ket.lb);
                               nq += l.t->quartets;
                               nq32 += fp32 ? l.t->quartets : 0.0;
                               fl += f;
                               queue.emplace_back(f, l);
                           };
                           for (int i = 0; i < static_cast<int>(c.cls.size()); i++)
                               for (int j = 0; j <= i; j++)
                               {
                                   if (c.cls[i].n_pairs == 0 || c.cls[j].n_pairs == 0)
                                       continue;
                                   add(i, j, mixed ? mixed_thresh : schwarz_thresh, kNoUpper, false);
                                   if (mixed)
                                       add(i, j, schwarz_thresh, mixed_thresh, true);
                               }
                           c.flushStaged();
                           std::stable_sort(queue.begin(), queue.end(),
                                            [](const auto &x, const auto &y) { return x.first > y.first; });
                           Fan fan(ctx->side, c.stream, queue.size() > 1);
                           for (auto &l : queue)
                           {
                               l.second.fn(l.second.a, fan.pick(l.first));
                               LBX_HIP(hipGetLastError());
                           }
                           fan.join();
                           hipLaunchKernelGGL(sumCopiesKernel, dim3(static_cast<int>((ng + 63) / 64)), dim3(64), 0,
                                              c.stream, ctx->grad_copies, grad, ng, lbx_context::kGradCopies);
                           LBX_HIP(hipGetLastError());
                           LBX_HIP(hipStreamSynchronize(c.stream));
                           if (stats)
                           {
                               stats->quartets = nq;
                               stats->flops = fl;
                               stats->quartets_fp32 = nq32;
                           }
                       });
    }

    int lbx_tune(lbx_context *ctx, const double *D, double schwarz_thresh)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx)
                               throw Error(LBX_ERR_INVALID, "lbx_tune: null argument");
                           if (!ctx->atom_mol.empty())
                           {
                               // a batched context: the RI sums' kernels (D is not used)
                               std::lock_guard<std::mutex> lk(ctx->mu);
                               if (ctx->shells_aux.empty())
                                   throw Error(LBX_ERR_STATE, "lbx_tune: the batched context has no auxiliary basis");
                               ctx->tuneRiSums();
                               return;
                           }
                           if (!D)
                               throw Error(LBX_ERR_INVALID, "lbx_tune: null argument");
                           if (!(schwarz_thresh >= 0))
                               throw Error(LBX_ERR_INVALID, "lbx_tune: negative Schwarz threshold");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           Context &c = *ctx;
                           ctx->ensureSchwarz();
                           const long long n = static_cast<long long>(c.nbf);
                           DevBuf J(n * n), K(n * n);
                           hipEvent_t e0, e1;
                           LBX_HIP(hipEventCreate(&e0));
                           LBX_HIP(hipEventCreate(&e1));
                           try
                           {
                               for (size_t i = 0; i < c.cls.size(); i++)
                                   for (size_t j = 0; j <= i; j++)
                                   {
                                       const PairClass &bra = c.cls[i], &ket = c.cls[j];
                                       if (bra.n_pairs == 0 || ket.n_pairs == 0)
                                           continue;
                                       int best = -1, best32 = -1;
                                       double best_ms = 0, best32_ms = 0;
                                       for (int v = 0; v < N_VARIANTS; v++)
                                       {
                                           if (!ownForm(v, kernelSlot(MODE_JK, bra.la, bra.lb, ket.la, ket.lb, v)))
                                               continue;
                                           if (isF32Variant(v))
                                               ensureF32(c);
                                           // first launch builds the task table and loads the code;
                                           // the timed one runs a sample of leading quartets
                                           ctx->sample_quartets = kTuneSample;
                                           if (ctx->launchJK(static_cast<int>(i), static_cast<int>(j), v, D, J.p, K.p,
                                                             schwarz_thresh) != v)
                                               continue;   // no room for its copy of E
                                           LBX_HIP(hipEventRecord(e0, c.stream));
                                           ctx->launchJK(static_cast<int>(i), static_cast<int>(j), v, D, J.p, K.p,
                                                         schwarz_thresh);
                                           LBX_HIP(hipEventRecord(e1, c.stream));
                                           ctx->sample_quartets = 0;
                                           LBX_HIP(hipEventSynchronize(e1));
                                           float ev = 0;
                                           LBX_HIP(hipEventElapsedTime(&ev, e0, e1));
                                           // time per quartet: the variants' samples differ
                                           const double ms = ev / std::max(ctx->sampled, 1.0);
                                           if (!isF32Variant(v) && (best < 0 || ms < best_ms))
                                           {
                                               best = v;
                                               best_ms = ms;
                                           }
                                           if (best32 < 0 || ms < best32_ms)
                                           {
                                               best32 = v;
                                               best32_ms = ms;
                                           }
                                       }
                                       ctx->dropJKGraphs();
                                       if (best >= 0)
                                           ctx->tuned[{static_cast<int>(i), static_cast<int>(j)}] = best;
                                       if (best32 >= 0)
                                           ctx->tuned32[{static_cast<int>(i), static_cast<int>(j)}] = best32;
                                   }
                           }
                           catch (...)
                           {
                               ctx->sample_quartets = 0;
                               (void)hipEventDestroy(e0);
                               (void)hipEventDestroy(e1);
                               throw;
                           }
                           ctx->sample_quartets = 0;
                           (void)hipEventDestroy(e0);
                           (void)hipEventDestroy(e1);
                           ctx->freeExtras();   // the forms that lost keep nothing
                       });
    }

    int lbx_set_variant(lbx_context *ctx, int la, int lb, int lc, int ld, int variant)
    {
        return guarded([&]
                       {
                           if (!ctx)
                               throw Error(LBX_ERR_INVALID, "lbx_set_variant: null context");
                           if (la < lb || lc < ld || la > kMaxLMain || lc > kMaxLMain || lb < 0 || ld < 0 ||
                               pairClassIdx(la, lb) < pairClassIdx(lc, ld))
                               throw Error(LBX_ERR_INVALID, "lbx_set_variant: not a canonical class pair");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           const std::pair<int, int> key{pairClassIdx(la, lb), pairClassIdx(lc, ld)};
                           ctx->dropJKGraphs();
                           if (variant < 0)
                           {
                               ctx->tuned.erase(key);
                               ctx->tuned32.erase(key);
                               return;
                           }
                           if (variant >= N_VARIANTS || !kernelSlot(MODE_JK, la, lb, lc, ld, variant).fn)
                               throw Error(LBX_ERR_INVALID, "lbx_set_variant: class pair has no such variant");
                           if (isF32Variant(variant))
                               ctx->tuned32[key] = variant;
                           else
                               ctx->tuned[key] = variant;
                       });
    }

    int lbx_set_class_filter(lbx_context *ctx, int la, int lb, int lc, int ld)
    {
        return guarded([&]
                       {
                           if (!ctx)
                               throw Error(LBX_ERR_INVALID, "lbx_set_class_filter: null context");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           if (la == -1 && lb == -1 && lc == -1 && ld == -1)
                           {
                               ctx->filter_i = ctx->filter_j = -1;
                               return;
                           }
                           if (la < lb || lc < ld || la > kMaxLMain || lc > kMaxLMain || lb < 0 || ld < 0 ||
                               pairClassIdx(la, lb) < pairClassIdx(lc, ld))
                               throw Error(LBX_ERR_INVALID, "lbx_set_class_filter: not a canonical class pair");
                           ctx->filter_i = pairClassIdx(la, lb);
                           ctx->filter_j = pairClassIdx(lc, ld);
                       });
    }

    int lbx_ri_jk(lbx_context *ctx, const double *D, double *J, double *K)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !D || !J)
                               throw Error(LBX_ERR_INVALID, "lbx_ri_jk: null argument");
                           long long n = 0, naux = 0;
                           hipStream_t s = nullptr;
                           {
                               std::lock_guard<std::mutex> lk(ctx->mu);
                               requireSingle(*ctx, "lbx_ri_jk");
                               if (ctx->shells_aux.empty())
                                   throw Error(LBX_ERR_STATE, "lbx_ri_jk: the context has no auxiliary basis");
                               n = static_cast<long long>(ctx->nbf);
                               naux = static_cast<long long>(ctx->nbf_aux);
                               s = ctx->stream;
                           }
                           riJK(ctx, *ctx, s, n, naux, D, J, K);
                       });
    }

    int lbx_one_electron(lbx_context *ctx, double *S, double *T, int ncharges, const double *charges, double *V)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || (!S && !T && !V))
                               throw Error(LBX_ERR_INVALID, "lbx_one_electron: null context or no output");
                           if (V && (ncharges < 0 || (ncharges > 0 && !charges)))
                               throw Error(LBX_ERR_INVALID, "lbx_one_electron: bad point charges");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           Context &c = *ctx;
                           requireSingle(c, "lbx_one_electron");
                           const size_t bytes = c.nbf * c.nbf * sizeof(double);
                           for (double *m : {S, T, V})
                               if (m)
                                   LBX_HIP(hipMemsetAsync(m, 0, bytes, c.stream));
                           double4 *d_q = nullptr;
                           if (V && ncharges > 0)
                           {
                               std::vector<double4> q(ncharges);
                               for (int k = 0; k < ncharges; k++)
                                   q[k] = double4{charges[4 * k], charges[4 * k + 1], charges[4 * k + 2],
                                                  charges[4 * k + 3]};
                               LBX_HIP(hipMalloc(&d_q, q.size() * sizeof(double4)));
                               const hipError_t e = hipMemcpyAsync(d_q, q.data(), q.size() * sizeof(double4),
                                                                   hipMemcpyHostToDevice, c.stream);
                               if (e != hipSuccess)
                               {
                                   (void)hipFree(d_q);
                                   LBX_HIP(e);
                               }
                           }
                           try
                           {
                               computeOneElectron(c, S, T, d_q, d_q ? ncharges : 0, V);
                               LBX_HIP(hipStreamSynchronize(c.stream));
                           }
                           catch (...)
                           {
                               (void)hipStreamSynchronize(c.stream);
                               (void)hipFree(d_q);
                               throw;
                           }
                           if (d_q)
                               LBX_HIP(hipFree(d_q));
                       });
    }

    int lbx_one_electron_grad(lbx_context *ctx, const double *D, const double *W, int ncharges,
                              const double *charges, double *grad, double *charge_grad)
    {
        return guardedIn(ctx, [&]
                       {
                           if (!ctx || !D || !grad)
                               throw Error(LBX_ERR_INVALID, "lbx_one_electron_grad: null argument");
                           if (ncharges < 0 || (ncharges > 0 && !charges))
                               throw Error(LBX_ERR_INVALID, "lbx_one_electron_grad: bad point charges");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           Context &c = *ctx;
                           requireSingle(c, "lbx_one_electron_grad");
                           LBX_HIP(hipMemsetAsync(grad, 0, static_cast<size_t>(c.natoms) * 3 * sizeof(double), c.stream));
                           if (charge_grad && ncharges > 0)
                               LBX_HIP(hipMemsetAsync(charge_grad, 0, static_cast<size_t>(ncharges) * 3 * sizeof(double),
                                                      c.stream));
                           double4 *d_q = nullptr;
                           if (ncharges > 0)
                           {
                               std::vector<double4> q(ncharges);
                               for (int k = 0; k < ncharges; k++)
                                   q[k] = double4{charges[4 * k], charges[4 * k + 1], charges[4 * k + 2],
                                                  charges[4 * k + 3]};
                               LBX_HIP(hipMalloc(&d_q, q.size() * sizeof(double4)));
                               const hipError_t e = hipMemcpyAsync(d_q, q.data(), q.size() * sizeof(double4),
                                                                   hipMemcpyHostToDevice, c.stream);
                               if (e != hipSuccess)
                               {
                                   (void)hipFree(d_q);
                                   LBX_HIP(e);
                               }
                           }
                           try
                           {
                               computeOneElectronGrad(c, D, W, d_q, ncharges, grad, charge_grad);
                           }
                           catch (...)
                           {
                               (void)hipStreamSynchronize(c.stream);
                               (void)hipFree(d_q);
                               throw;
                           }
                           if (d_q)
                               LBX_HIP(hipFree(d_q));
                       });
    }

    int lbx_set_bound_window(lbx_context *ctx, double lo, double hi)
    {
        return guarded([&]
                       {
                           if (!ctx)
                               throw Error(LBX_ERR_INVALID, "lbx_set_bound_window: null context");
                           if (!(lo >= 0.0) || !(hi > lo))
                               throw Error(LBX_ERR_INVALID, "lbx_set_bound_window: need 0 <= lo < hi");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           ctx->window_lo = lo;
                           ctx->window_hi = hi;
                       });
    }

    int lbx_profile_enable(lbx_context *ctx, int on)
    {
        return guarded([&]
                       {
                           if (!ctx)
                               throw Error(LBX_ERR_INVALID, "lbx_profile_enable: null context");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           if (on)
                               for (auto &kv : ctx->prof)
                               {
                                   lbx_class_profile keep = kv.second.rec;
                                   kv.second.rec = lbx_class_profile{};
                                   kv.second.rec.la = keep.la;
                                   kv.second.rec.lb = keep.lb;
                                   kv.second.rec.lc = keep.lc;
                                   kv.second.rec.ld = keep.ld;
                                   kv.second.rec.kernel = keep.kernel;
                                   kv.second.pending = false;
                               }
                           ctx->profiling = on != 0;
                       });
    }

    int lbx_profile_read(lbx_context *ctx, lbx_class_profile *out, int capacity, int *count)
    {
        return guarded([&]
                       {
                           if (!ctx || !count || (capacity > 0 && !out))
                               throw Error(LBX_ERR_INVALID, "lbx_profile_read: null argument");
                           std::lock_guard<std::mutex> lk(ctx->mu);
                           int n = 0;
                           for (auto &kv : ctx->prof)
                           {
                               if (kv.second.rec.calls == 0)
                                   continue;
                               if (n < capacity)
                                   out[n] = kv.second.rec;
                               n++;
                           }
                           *count = n;
                       });
    }
}
