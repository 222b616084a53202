// autotune.cpp -- per-size choice of solver, precision and pair-kernel rows per workgroup, measured
// on the GPU it runs on and cached.
//
// The reference fixes its launch shapes (16 x 16 threads per matrix block, 256 per vector kernel,
// BoundaryProblem.cuh:27-34) and always solves with getrf/getrs (MatrixSolver.cuh:113-172).  Here the
// right choice depends on N: the blocked LU is a serial chain of panels, GMRES a few launches bound by their
// latency (small N) or by FP64 issue (large N), the persistent batched kernel suits N <= 1024, and a workgroup of
// 4 rows leaves most CUs idle when N / 4 is well below the CU count.  autotune() times each candidate on a seeded 8-mode surface
// of the handle's physics (warm-up through the GMRES calibration, then timed steps replayed from the
// step graph), rejects candidates whose solves do not converge, and keeps the fastest.  Options that the launched
// kernels do not depend on are not tried (candidates()).  Results are
// cached per (GPU architecture, problem kind, image term and GMRES route, N, mixed allowed) in memory and in a text
// file: $SFH_TUNE_CACHE, else $XDG_CACHE_HOME/cusuperhelium/tuning.txt, else
// $HOME/.cache/cusuperhelium/tuning.txt (memory only when none is writable).
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <map>
#include <mutex>
#include <random>
#include <sstream>
#include <string>
#include <sys/stat.h>
#include <tuple>
#include <vector>

#include "sfh_gmres.hpp"
#include "solver.hpp"

namespace sfh {

namespace {

std::mutex g_tune_mu;
std::map<std::string, Tuning> g_tunings;
bool g_file_loaded = false;

std::string arch_name() {
    int dev = 0;
    SFH_HIP(hipGetDevice(&dev));
    hipDeviceProp_t p;
    SFH_HIP(hipGetDeviceProperties(&p, dev));
    std::string a = p.gcnArchName;
    for (char& c : a)
        if (c == ' ' || c == ':') c = '_';
    return a.empty() ? std::string("unknown") : a;
}

// The first field carries the version of the kernels that were timed: entries of other versions match no key.  The third
// is the image term (1), plus 2 where GMRES stores its matrix (rho quirk, thin films) and is another candidate.
constexpr const char* kTuneVersion = "/2";

int route_of(const Phys& ph, int n) { return (ph.image ? 1 : 0) + (gmres_sums(ph, n, kGmMaxIter) ? 0 : 2); }

std::string key_of(const std::string& arch, int kind, int route, int n, bool mixed) {
    std::ostringstream k;
    k << arch << ' ' << kind << ' ' << route << ' ' << n << ' ' << (mixed ? 1 : 0);
    return k.str();
}
std::string key_of(const Phys& ph, int n, bool mixed) {
    return key_of(arch_name() + kTuneVersion, ph.kind, route_of(ph, n), n, mixed);
}

std::string cache_path() {
    if (const char* p = std::getenv("SFH_TUNE_CACHE")) return p;
    std::string base;
    if (const char* x = std::getenv("XDG_CACHE_HOME")) base = x;
    else if (const char* h = std::getenv("HOME")) base = std::string(h) + "/.cache";
    else return "";
    return base + "/cusuperhelium/tuning.txt";
}

void load_file() {
    if (g_file_loaded) return;
    g_file_loaded = true;
    const std::string path = cache_path();
    if (path.empty()) return;
    std::ifstream in(path);
    std::string line;
    while (std::getline(in, line)) {
        if (line.empty() || line[0] == '#') continue;
        std::istringstream ls(line);
        std::string arch;
        int kind, route, n, mixed;
        Tuning t;
        if (ls >> arch >> kind >> route >> n >> mixed >> t.solver >> t.precision >> t.pair_rows >> t.ms_per_step)
            g_tunings[key_of(arch, kind, route, n, mixed != 0)] = t;
    }
}

void save_file() {
    const std::string path = cache_path();
    if (path.empty()) return;
    const size_t slash = path.rfind('/');
    if (slash != std::string::npos) {   // create the directory chain
        std::string dir = path.substr(0, slash);
        for (size_t i = 1; i <= dir.size(); ++i)
            if (i == dir.size() || dir[i] == '/') mkdir(dir.substr(0, i).c_str(), 0755);
    }
    const std::string tmp = path + ".tmp" + std::to_string((long long)std::rand());
    {
        std::ofstream out(tmp);
        if (!out) return;
        out << "# arch/version kind image+2*stored n mixed_allowed solver precision pair_rows ms_per_step\n";
        for (const auto& kv : g_tunings) {
            const Tuning& t = kv.second;
            out << kv.first << ' ' << t.solver << ' ' << t.precision << ' ' << t.pair_rows << ' ' << t.ms_per_step
                << '\n';
        }
    }
    std::rename(tmp.c_str(), path.c_str());
}

// the 8-mode seeded surface of the benchmark workloads (a_k ~ U(0, 0.02/k), phases uniform)
void probe_state(int n, std::vector<double>& x, std::vector<double>& y, std::vector<double>& p) {
    std::mt19937_64 rng(20261202u + (unsigned)n);
    std::uniform_real_distribution<double> u(0.0, 1.0);
    double a[8], th[8];
    for (int k = 0; k < 8; ++k) {
        a[k] = 0.02 / (k + 1) * u(rng);
        th[k] = 2.0 * kPi * u(rng);
    }
    x.resize(n);
    y.resize(n);
    p.assign(n, 0.0);
    for (int j = 0; j < n; ++j) {
        x[j] = 2.0 * kPi * j / n;
        double s = 0.0;
        for (int k = 0; k < 8; ++k) s += a[k] * std::cos((k + 1) * x[j] + th[k]);
        y[j] = s;
    }
}

// ms per step of one candidate, or +inf if it fails or leaves a solve unconverged
double time_candidate(const Phys& ph, int n, const Options& o, int steps, const std::vector<double>& x,
                      const std::vector<double>& y, const std::vector<double>& p) {
    try {
        Solver s(ph, std::vector<int>(1, n), o);
        s.set_state(x.data(), y.data(), p.data());
        const double dt = 0.002;
        s.step(dt, 8);   // warm-up: graph capture, warm-start history, GMRES calibration
        s.sync();
        const auto t0 = std::chrono::steady_clock::now();
        s.step(dt, steps);
        s.sync();
        const auto t1 = std::chrono::steady_clock::now();
        if (s.stats().unconverged) return INFINITY;
        return std::chrono::duration<double, std::milli>(t1 - t0).count() / steps;
    } catch (const std::exception&) {
        return INFINITY;
    }
}

struct Cand {
    int solver, precision, rows;
};

// The forms that differ in what they launch.  Rows per workgroup of the pair kernels matter to LU above 256 nodes and
// with the rho quirk, and to GMRES with a stored matrix; the mixed form of GMRES only where that matrix is FP32 (water).
std::vector<Cand> candidates(const Phys& ph, int n, bool allow_mixed) {
    const bool quirk = ph.kind == 0 && ph.rho_quirk && ph.rho != 0.0;
    const bool stored = !gmres_sums(ph, n, kGmMaxIter);
    std::vector<Cand> c;
    for (int rows : {1, 2, 4}) {
        if (rows == kPairRows || n > kSmallNodes || quirk) c.push_back({kSolveLU, kFP64, rows});
        if (n <= kGmMaxN && (rows == kPairRows || stored)) {
            c.push_back({kSolveGMRES, kFP64, rows});
            if (allow_mixed && stored && !ph.image) c.push_back({kSolveGMRES, kMixed, rows});
        }
    }
    if (n <= kBatchMaxN) {
        c.push_back({kSolveBatched, kFP64, kPairRows});
        if (allow_mixed) c.push_back({kSolveBatched, kMixed, kPairRows});
    }
    return c;
}

}  // namespace

Tuning autotune(const Phys& ph_in, int n, bool allow_mixed, int steps) {
    if (!supported_n(n)) throw ArgError("unsupported node count " + std::to_string(n));
    if (steps < 1) throw ArgError("steps must be positive");
    Phys ph = ph_in;
    ph.drive = ph.augmented = 0;   // the drive's per-node epilogue does not change the ranking
    std::vector<double> x, y, p;
    probe_state(n, x, y, p);
    Tuning best;
    best.ms_per_step = INFINITY;
    for (const Cand& c : candidates(ph, n, allow_mixed)) {
        Options o;
        o.solver = c.solver;
        o.precision = c.precision;
        o.pair_rows = c.rows;
        o.max_iter = c.solver == kSolveBatched ? 16 : kGmMaxIter;
        const double ms = time_candidate(ph, n, o, steps, x, y, p);
        if (ms < best.ms_per_step) {
            best.solver = c.solver;
            best.precision = c.precision;
            best.pair_rows = c.rows;
            best.ms_per_step = ms;
        }
    }
    if (!std::isfinite(best.ms_per_step)) throw HipError("autotune: no candidate ran");
    std::lock_guard<std::mutex> lk(g_tune_mu);
    load_file();
    g_tunings[key_of(ph, n, allow_mixed)] = best;
    save_file();
    best.from_cache = 0;
    return best;
}

Tuning tuned(const Phys& ph, int n, bool allow_mixed) {
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        load_file();
        auto it = g_tunings.find(key_of(ph, n, allow_mixed));
        if (it != g_tunings.end()) {
            Tuning t = it->second;
            t.from_cache = 1;
            return t;
        }
    }
    return autotune(ph, n, allow_mixed, 10);
}

}  // namespace sfh
