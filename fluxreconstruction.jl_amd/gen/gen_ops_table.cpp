// gen_ops_table.cpp -- writes csrc/fr_ops_table.h: the 2D kernel operators (Gauss-Legendre
// solution points, Radau correction; the pair FRPSpace2D hard-wires at src/struct.jl:193) of
// degrees 1..5 and the 1D operators that do not depend on the correction function, degrees 1..8, as
// compile-time constants, taken bit for bit from the library's build_ops.
//   usage: gen_ops_table > csrc/fr_ops_table.h
#include <cstdio>

#include "../csrc/fr_common.h"

static void arr(const char *name, const double *v, int n) {
  std::printf("  static constexpr double %s[%d] = {", name, n);
  for (int i = 0; i < n; ++i) std::printf("%s%a", i ? ", " : "", v[i]);
  std::printf("};\n");
}

int main() {
  std::printf("// fr_ops_table.h -- generated by gen/gen_ops_table.cpp from fr::build_ops (Gauss-Legendre\n"
              "// points, Radau correction); do not edit.  dl is column-major: dl[k + nsp*q] = l_q'(r_k);\n"
              "// dc[k + nsp*q] = dl[k + nsp*q] - ll[q]*dhl[k] - lr[q]*dhr[k] is the derivative with the\n"
              "// flux-trace parts of both correction terms folded in (rounded once from long double).\n"
              "// StdOps1D: hw are half the Gauss weights (they sum to one), V1 and iV1 the modal matrix and\n"
              "// its inverse, column-major.\n"
              "#pragma once\n\nnamespace fr {\n\ntemplate <int NSP>\nstruct StdOps2D;\n");
  for (int deg = 1; deg <= 5; ++deg) {
    fr::HostOps o;
    if (!fr::build_ops(deg, FR_CORR_RADAU, o)) return 1;
    const int n = deg + 1;
    std::printf("\ntemplate <>\nstruct StdOps2D<%d> {\n", n);
    arr("ll", o.ll, n);
    arr("lr", o.lr, n);
    arr("dl", o.dl, n * n);
    arr("dhl", o.dhl, n);
    arr("dhr", o.dhr, n);
    double dc[64];
    for (int q = 0; q < n; ++q)
      for (int k = 0; k < n; ++k)
        dc[k + n * q] = (double)((long double)o.dl[k + n * q] - (long double)o.ll[q] * (long double)o.dhl[k] -
                                 (long double)o.lr[q] * (long double)o.dhr[k]);
    arr("dc", dc, n * n);
    std::printf("};\n");
  }
  std::printf("\ntemplate <int NSP>\nstruct StdOps1D;\n");
  for (int deg = 1; deg <= 8; ++deg) {
    fr::HostOps o;
    if (!fr::build_ops(deg, FR_CORR_RADAU, o)) return 1;
    const int n = deg + 1;
    std::printf("\ntemplate <>\nstruct StdOps1D<%d> {\n", n);
    arr("ll", o.ll, n);
    arr("lr", o.lr, n);
    arr("dl", o.dl, n * n);
    double hw[16];
    for (int q = 0; q < n; ++q) hw[q] = 0.5 * o.w[q];
    arr("hw", hw, n);
    arr("V1", o.V1, n * n);
    arr("iV1", o.iV1, n * n);
    std::printf("};\n");
  }
  std::printf("\n}  // namespace fr\n");
  return 0;
}
