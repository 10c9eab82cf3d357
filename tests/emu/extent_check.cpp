// TEST-ONLY: the stage kernels' index arithmetic at the largest accepted
// problem (n = 2048), compiled for the CPU against the shim.  One tile of panel
// 1 and the same tile of panel 6, with the same values at its points, run in
// full-size arrays: sparse mappings of which only the tile's pages exist, zero
// everywhere else.  Panel 1 keeps every byte offset small, so an offset that
// wraps on panel 6 (where they are largest) reads other values or leaves its
// results elsewhere, and the two panels differ.  Exit status 0: none did.
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../mcv_sw_amd/csrc/mcv_fp32c.hpp"
#include "../../mcv_sw_amd/csrc/mcv_stage_fp64.hpp"

using namespace mcv;

// `count` elements, zero, taking memory only where written.
template <typename T>
struct Sparse {
  T *p;
  size_t count;
  explicit Sparse(size_t n) : count(n) {
    void *m = mmap(nullptr, n * sizeof(T), PROT_READ | PROT_WRITE,
                   MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) {
      std::perror("mmap");
      std::exit(2);
    }
    p = static_cast<T *>(m);
  }
  ~Sparse() { munmap(p, count * sizeof(T)); }
  operator T *() const { return p; }
};

static int g_bad = 0;

static void same(const char *what, const void *a, const void *b, size_t bytes) {
  static const char zero[64] = {};
  if (std::memcmp(a, b, bytes) != 0 || std::memcmp(a, zero, bytes) == 0) {
    if (++g_bad <= 20) std::printf("  %s: panel 6 differs from panel 1, or nothing was written\n", what);
  }
}

// A value of its own for every (array k, point q).
static double val(int k, long long q) { return 1.0 + 1e-3 * k + 1e-6 * (double)(q % 9973); }

struct Tile {
  int i0, j0, lw, lh, ox, oy;  // first core point, staged extents, owned extents
};

static Tile tile_of(int dof, int n, int CX, int CY, int tx, int ty) {
  const int H = dof - 1, cx0 = tx * CX, cy0 = ty * CY;
  const int ncx = std::min(CX, n - cx0), ncy = std::min(CY, n - cy0);
  return Tile{cx0 * H + 1, cy0 * H + 1, ncx * H + 1 + 2 * H, ncy * H + 1 + 2 * H,
              ncx * H + (cx0 + ncx == n), ncy * H + (cy0 + ncy == n)};
}

// One tile on panels 1 and 6 in the arrays of an n^2 problem.
template <int DOF, int CX, int CY, bool F32>
static void check(int n, int kind, bool far) {
  constexpr int H = DOF - 1;
  const int npv = n * H + 1, nh = npv + 2 * H;
  const size_t per = (size_t)nh * nh, np = 6 * per;
  const int tx = far ? (n + CX - 1) / CX - 1 : 0, ty = far ? (n + CY - 1) / CY - 1 : 0;
  const Tile t = tile_of(DOF, n, CX, CY, tx, ty);
  // per panel, so that panel 6 has metric terms of its own too
  Sparse<D2> mpack(2 * np);
  Sparse<double> p2sp(4 * np), f(np), phis(np);
  Sparse<D3> band(band_points(DOF, npv));
  const size_t nt = (size_t)6 * npv * npv;
  std::vector<char> smem(160 * 1024 + 64);
  char *const lds = smem.data() + (64 - (uintptr_t)smem.data() % 64) % 64;
  auto points = [&](auto &&put) {  // the staged points of both panels
    for (int p : {1, 6})
      for (int ly = 0; ly < t.lh; ++ly)
        for (int lx = 0; lx < t.lw; ++lx) put(pidx(nh, H, p, t.i0 - H + lx, t.j0 - H + ly), ly * t.lw + lx);
  };
  points([&](long long g, int q) {
    mpack[2 * g] = D2{val(0, q), 1.0};
    mpack[2 * g + 1] = D2{0.1 * val(1, q), val(2, q)};
    for (int k = 0; k < 4; ++k) p2sp[4 * g + k] = val(3 + k, q);
    f[g] = 1e-4 * val(7, q);
    phis[g] = 10.0 * val(8, q);
  });
  const double dx = 1e-3;
  // every owned point: results in the same words of the two panels
  auto owned = [&](auto &&cmp) {
    for (int y = 0; y < t.oy; ++y)
      for (int x = 0; x < t.ox; ++x) {
        const int i = t.i0 + x, j = t.j0 + y;
        cmp(pidx(nh, H, 1, i, j), pidx(nh, H, 6, i, j),
            ((size_t)(j - 1) * npv + (i - 1)), ((size_t)(5 * (size_t)npv + j - 1) * npv + (i - 1)));
        if (kind == kTend) continue;
        for (int s = 0; s < 4; ++s)
          for (int d = 1; d <= H + 1; ++d) {
            const int al = s < 2 ? j : i;
            int bi, bj;
            band_ij(npv, s, d, al, bi, bj);
            if (bi == i && bj == j)
              same("band", &band[band_point(npv, H, 1, s, d, al)],
                   &band[band_point(npv, H, 6, s, d, al)], sizeof(D3));
          }
      }
  };
  if constexpr (!F32) {
    Sparse<D2> in(np), base(np), acc(np), out(kind == kTend ? nt : np);
    Sparse<double> in_v(np), base_v(np), acc_v(np), out_v(kind == kTend ? nt : np), cu(np), cv(np);
    points([&](long long g, int q) {
      in[g] = D2{5e4 * val(10, q), val(11, q)};
      in_v[g] = val(12, q);
      base[g] = D2{5e4 * val(13, q), val(14, q)};
      base_v[g] = val(15, q);
      acc[g] = D2{val(16, q), val(17, q)};
      acc_v[g] = val(18, q);
      cu[g] = val(19, q);
      cv[g] = val(20, q);
    });
    MeshDev m{};
    m.dof = DOF; m.n = n; m.npv = npv; m.nh = nh; m.dx = dx;
    m.dv = MCVDivisors{make_recip(dx), make_recip(2 * dx), make_recip(dx * dx)};
    m.metric_pstride = m.phis_pstride = (long long)per;
    m.mpack = mpack; m.f = f; m.phi_s = phis; m.p2sp = p2sp;
    StageArgs a{};
    a.in_pu = in; a.in_v = in_v; a.b_pu = base; a.b_v = base_v; a.acc_pu = acc; a.acc_v = acc_v;
    a.o_pu = out; a.o_v = out_v; a.band_raw = band; a.cu0 = cu; a.cv0 = cv; a.c1 = 1.0;
    for (int p : {1, 6})
      stage_body<DOF, CX, CY>(m, a, kind, false, kind == kTend || kind == kRK4S1, p, tx, ty, lds);
    owned([&](long long a1, long long a6, size_t t1, size_t t6) {
      const size_t o1 = kind == kTend ? t1 : a1, o6 = kind == kTend ? t6 : a6;
      same("phi, u", &out[o1], &out[o6], sizeof(D2));
      same("v", &out_v[o1], &out_v[o6], sizeof(double));
      same("accumulator", &acc[a1], &acc[a6], sizeof(D2));
      same("accumulator v", &acc_v[a1], &acc_v[a6], sizeof(double));
    });
  } else {
    Sparse<F3> in(np), base(np), comp(np), acc(np), out(np), oc(np);
    Sparse<double> pgref(np);
    Sparse<F4> fdE(np);
    points([&](long long g, int q) {
      in[g] = F3{(float)val(10, q), (float)val(11, q), (float)val(12, q)};
      base[g] = F3{(float)val(13, q), (float)val(14, q), (float)val(15, q)};
      comp[g] = F3{1e-8f * (float)val(16, q), 1e-8f, 2e-8f};
      acc[g] = F3{(float)val(17, q), (float)val(18, q), (float)val(19, q)};
      pgref[g] = 5e4 * val(20, q);
      fdE[g] = F4{(float)val(21, q), (float)val(22, q), 1e-4f, 0.f};
    });
    MeshF32 m{};
    m.dof = DOF; m.n = n; m.npv = npv; m.nh = nh;
    m.rdx = 1 / dx; m.r2dx = 1 / (2 * dx); m.rdxx = 1 / (dx * dx); m.dx = dx;
    m.metric_pstride = (long long)per;
    m.mpack = mpack; m.pgref = pgref; m.fdE = fdE; m.p2sp = p2sp;
    const bool last = kind == kRK4S4 || kind == kRK3S3;
    StageArgs32 a{};
    a.in = in; a.b = base; a.c = comp; a.acc = acc; a.o = out; a.oc = last ? oc.p : nullptr;
    a.band_raw = band; a.c1 = 1.0;
    for (int p : {1, 6}) stage_body_f32<DOF, CX, CY>(m, a, kind, false, p, tx, ty, lds);
    owned([&](long long a1, long long a6, size_t, size_t) {
      same("level", &out[a1], &out[a6], sizeof(F3));
      if (last) same("compensation", &oc[a1], &oc[a6], sizeof(F3));
      same("accumulator", &acc[a1], &acc[a6], sizeof(F3));
    });
  }
}

template <int DOF, int CX, int CY>
static void all(int n) {
  for (bool far : {false, true}) {
    for (int kind : {kTend, kRK4S1, kRK4S2, kRK4S4, kRK3S3}) {
      std::printf("MCV%d FP64 kind %d %s\n", DOF, kind, far ? "far corner" : "near corner");
      check<DOF, CX, CY, false>(n, kind, far);
    }
    for (int kind : {kRK4S1, kRK4S2, kRK4S4, kRK3S3}) {
      std::printf("MCV%d FP32C kind %d %s\n", DOF, kind, far ? "far corner" : "near corner");
      check<DOF, CX, CY, true>(n, kind, far);
    }
  }
}

int main() {
  const int n = 2048;
  all<3, 8, 7>(n);
  all<4, 6, 4>(n);
  if (g_bad) std::printf("%d differences\n", g_bad);
  return g_bad ? 1 : 0;
}
