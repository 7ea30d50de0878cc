// Where the one-pass step looks for psi, against pml_face's own index: for
// each grid given as nx,ny,nz,layers,value bytes, every face of both passes at
// the corners of its corrected nodes and at random ones.  Prints, per grid,
// the faces that 32-bit offsets reach, the faces in all, and the nodes whose
// address differs on a face said to be reached.
#include <cinttypes>
#include <cstdio>
#include <cstdlib>
#include <random>

#include "../../xfdtd_cuda_amd/csrc/xf_kernels.h"

namespace {

template <typename C>
void grid(int64_t nx, int64_t ny, int64_t nz, int64_t layers) {
  const int64_t n[3] = {nx, ny, nz};
  std::mt19937_64 rng(1);
  int reached = 0, faces = 0;
  int64_t wrong = 0;
  for (int f = 0; f < 6; ++f)
    for (int pass = 0; pass < 2; ++pass) {
      const bool is_e = pass == 1, high = f & 1;
      const int ax = f / 2, la = (ax + 1) % 3, lb = (ax + 2) % 3;
      xf::PmlFace<C> F{};
      F.axis = ax;
      const int64_t cs = high ? n[ax] - layers : 0;
      const int64_t off = is_e && cs == 0 ? 1 : 0;
      F.c0 = static_cast<int>(cs + off);
      F.c1 = static_cast<int>(cs + layers + off);
      F.a0 = F.b0 = 0;
      F.a1 = static_cast<int>(n[la]);
      F.b1 = static_cast<int>(n[lb]);
      F.nstart = F.c0;
      // lateral sizes of psi_a and psi_b: one axis has a node more
      const auto shape = [&](bool a_closed, int64_t* s1, int64_t* s2) {
        int64_t s[3];
        s[ax] = layers;
        s[la] = n[la] + (a_closed ? 1 : 0);
        s[lb] = n[lb] + (a_closed ? 0 : 1);
        *s1 = s[1];
        *s2 = s[2];
      };
      shape(!is_e, &F.sa1, &F.sa2);
      shape(is_e, &F.sb1, &F.sb2);
      // addresses are compared, never used
      F.psi_a = reinterpret_cast<C*>(uint64_t(1) << 44);
      F.psi_b = reinterpret_cast<C*>(uint64_t(2) << 44);
      F.cpsi_a = reinterpret_cast<C*>(uint64_t(3) << 44);
      F.cpsi_b = reinterpret_cast<C*>(uint64_t(4) << 44);
      C* const oa = reinterpret_cast<C*>(uint64_t(5) << 44);
      C* const ob = reinterpret_cast<C*>(uint64_t(6) << 44);
      const xf::Step3Face<C> D = xf::step3_face<C>(F, is_e, oa, ob);
      ++faces;
      if (!xf::step3_face_fits(D)) continue;
      ++reached;
      const auto node = [&](int64_t a, int64_t b, int64_t c) {
        int64_t at[3];
        at[ax] = c;
        at[la] = a;
        at[lb] = b;
        const int64_t layer = c - F.nstart;
        const int64_t px = ax == 0 ? layer : ax == 1 ? b : a, py = ax == 0 ? a : ax == 1 ? layer : b,
                      pz = ax == 0 ? b : ax == 1 ? a : layer;
        const bool in_a = is_e ? a < F.a1 : b < F.b1, in_b = is_e ? b < F.b1 : a < F.a1;
        const int i = static_cast<int>(at[0]), j = static_cast<int>(at[1]), k = static_cast<int>(at[2]);
        const auto same = [&](const C* biased, const C* array, uint32_t offset, int64_t index) {
          if (reinterpret_cast<uint64_t>(biased) + offset != reinterpret_cast<uint64_t>(array) + index * sizeof(C)) ++wrong;
        };
        if (in_a) {
          const uint32_t o = xf::step3_psi_offset<C>(i, j, k, D.lo, D.row_a, D.plane_a);
          const int64_t p = (px * F.sa1 + py) * F.sa2 + pz;
          same(D.a, F.psi_a, o, p);
          same(D.oa, oa, o, p);
          same(D.cpa, F.cpsi_a, o, p);
        }
        if (in_b) {
          const uint32_t o = xf::step3_psi_offset<C>(i, j, k, D.lo, D.row_b, D.plane_b);
          const int64_t p = (px * F.sb1 + py) * F.sb2 + pz;
          same(D.b, F.psi_b, o, p);
          same(D.ob, ob, o, p);
          same(D.cpb, F.cpsi_b, o, p);
        }
      };
      for (int64_t a : {int64_t(0), int64_t(F.a1)})
        for (int64_t b : {int64_t(0), int64_t(F.b1)})
          for (int64_t c : {int64_t(F.c0), int64_t(F.c1) - 1}) node(a, b, c);
      for (int q = 0; q < 2000; ++q) {
        const int64_t a = static_cast<int64_t>(rng() % (F.a1 + 1)), b = static_cast<int64_t>(rng() % (F.b1 + 1));
        node(a, b, F.c0 + static_cast<int64_t>(rng() % (F.c1 - F.c0)));
      }
    }
  std::printf("%d %d %" PRId64 "\n", reached, faces, wrong);
}

}  // namespace

int main(int argc, char** argv) {
  for (int q = 1; q < argc; ++q) {
    long long v[5];
    if (std::sscanf(argv[q], "%lld,%lld,%lld,%lld,%lld", v, v + 1, v + 2, v + 3, v + 4) != 5) return 2;
    if (v[4] == 8)
      grid<double>(v[0], v[1], v[2], v[3]);
    else
      grid<float>(v[0], v[1], v[2], v[3]);
  }
  return 0;
}
