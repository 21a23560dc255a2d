// fast_shim.cpp -- TEST INFRASTRUCTURE.  A host-only build of the face physics
// (harm_device.h), of its shorter form (harm_fast.h) and of the serial sum by
// runs (harm_chain.h), so that the CPU tests can compare them with the plain
// forms.  Built by the tests with
//   hipcc -x hip --offload-host-only -O2 -ffp-contract=off -shared -fPIC
#include "../harm_ramt_amd/csrc/harm_chain.h"
#include "../harm_ramt_amd/csrc/harm_fast.h"

using namespace harm;

static KParams mkP(const double* prm) {
  // prm: gam, eomtype, fluxmethod, gammamax, lim, cour, dx1, dx2
  KParams P = {};
  P.gam = prm[0];
  P.eomtype = (int)prm[1];
  P.fluxmethod = (int)prm[2];
  P.gammamax = prm[3];
  P.lim = (int)prm[4];
  P.cour = prm[5];
  P.dx1 = prm[6];
  P.dx2 = prm[7];
  return P;
}

extern "C" {

// n faces of direction dir: geo [n][16] (gcov upper 10, gcon^{00..03},
// gcon^{dd}, gdet), pl, pr [n][8].  general, fast: F [n][8] and [n] Courant
// limits; fail [n][2]; ok[n]: the shorter form holds
void shim_faces(const double* prm, int dir, long n, const double* geo, const double* pl, const double* pr,
                double* Fgen, double* dtgen, double* Ffast, double* dtfast, int* fail, int* ok) {
  const KParams P = mkP(prm);
  for (long m = 0; m < n; m++) {
    const double* a = geo + m * 16;
    GeoU g;
    g.g00 = a[0]; g.g01 = a[1]; g.g02 = a[2]; g.g03 = a[3]; g.g11 = a[4]; g.g12 = a[5];
    g.g13 = a[6]; g.g22 = a[7]; g.g23 = a[8]; g.g33 = a[9];
    g.n00 = a[10]; g.n01 = a[11]; g.n02 = a[12]; g.n03 = a[13]; g.ndd = a[14]; g.gdet = a[15];
    double l[NPR], r[NPR], Fo[NPR], cm = 0.;
    for (int k = 0; k < NPR; k++) {
      l[k] = pl[m * 8 + k];
      r[k] = pr[m * 8 + k];
    }
    fail[2 * m] = fail[2 * m + 1] = 0;
    ok[m] = (dir == 1) ? face_flux_fast<1>(P, l, r, g, Fo, cm, fail[2 * m + 1])
                       : face_flux_fast<2>(P, l, r, g, Fo, cm, fail[2 * m + 1]);
    for (int k = 0; k < NPR; k++) Ffast[m * 8 + k] = Fo[k];
    const double d = P.cour * ((dir == 1) ? P.dx1 : P.dx2) / cm;
    dtfast[m] = (d < 1.e9) ? d : 1.e9;
    if (dir == 1) face_flux<1>(P, l, r, g, Fgen + m * 8, dtgen[m], fail[2 * m]);
    else face_flux<2>(P, l, r, g, Fgen + m * 8, dtgen[m], fail[2 * m]);
  }
}

// n five-zone stencils y [n][5]: edges [n][2] of para4 and of para4_fast, and
// whether the latter's finiteness sum holds
void shim_para4(long n, const double* y, double* gen, double* fast, int* ok) {
  for (long m = 0; m < n; m++) {
    const double* a = y + m * 5;
    double z = 0.;
    para4(a[0], a[1], a[2], a[3], a[4], gen[2 * m], gen[2 * m + 1]);
    para4_fast(a[0], a[1], a[2], a[3], a[4], fast[2 * m], fast[2 * m + 1], z);
    ok[m] = (z == 0.);
  }
}

// n quotients by the shared-reciprocal steps: q[m] = a[m] / d[m]
void shim_quotients(long n, const double* a, const double* d, double* q) {
  for (long m = 0; m < n; m++) {
    const double num[1] = {a[m]};
    double out[1];
    Divisor(d[m]).under(num, out);
    q[m] = out[0];
  }
}

// the sum s + t[0] + t[1] + ... (n a multiple of 16) by runs of 16, their maps
// composed from each start on as a scan does; *by_map: the runs whose map held
double shim_chain(long n, const double* t, double s, long* by_map) {
  const long runs = n / 16;
  *by_map = 0;
  for (long r = 0; r < runs;) {
    const ChainScale c(s);
    double d0 = 0., d1 = 0.;
    int q = 2;
    long k = r;
    if (c.e >= 0)
      for (; k < runs; k++) {
        double v[16];
        memcpy(v, t + 16 * k, sizeof(v));
        ChainMap m = chain_map(c, v);
        const double at = fabs(s) + ((chain_bits(s) & 1) ? d1 : d0);
        if (!chain_holds(c, at, m.mn, m.mx)) break;
        double a0 = m.d0, a1 = m.d1;
        int aq = m.q;
        chain_then(d0, d1, q, a0, a1, aq);
        d0 = a0;
        d1 = a1;
        q = aq;
      }
    *by_map += k - r;
    if (k > r) {
      const double end = fabs(s) + ((chain_bits(s) & 1) ? d1 : d0);
      s = (chain_bits(s) >> 63) ? -end : end;
    }
    if (k < runs)
      for (int m = 0; m < 16; m++) s += t[16 * k + m];
    r = k + 1;
  }
  return s;
}

}
