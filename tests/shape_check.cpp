// Test support: compile a form's kernels for gfx950 without a GPU under given
// shape options (description as in codegen_check.cpp), built by
// tests/test_shapes_cpu.py against the library's object files.
//
//   shape_check <description> <out.co> [<option>=<value>...]
//
// Prints "OK", or "FAIL <message>".
#include <cstdlib>
#include <fstream>
#include <iostream>
#include <memory>
#include <string>

#include "mf_internal.h"

int main(int argc, char** argv) {
  try {
    if (argc < 3) throw std::runtime_error("usage: shape_check <description> <out.co> [<option>=<value>...]");
    std::ifstream in(argv[1]);
    int rank, nv, nf, W, nd0, bs0, nd1, bs1, nint, ncoef;
    in >> rank >> nv >> nf >> W >> nd0 >> bs0 >> nd1 >> bs1 >> nint >> ncoef;
    mf_mesh mesh;
    mf_dofmap dm0, dm1;
    mf_form f;
    mesh.nv = nv;
    mesh.nf = nf;
    dm0.nd = nd0;
    dm0.bs = bs0;
    dm1.nd = nd1;
    dm1.bs = bs1;
    f.rank = rank;
    f.mesh = &mesh;
    f.dm[0] = rank >= 1 ? &dm0 : nullptr;
    f.dm[1] = rank == 2 ? (nd0 == nd1 && bs0 == bs1 ? &dm0 : &dm1) : nullptr;
    f.W = W;
    for (int c = 0; c < ncoef; ++c) {
      mf::Coef co;
      in >> co.offset >> co.width;
      f.coefs.push_back(std::move(co));
    }
    for (int i = 0; i < nint; ++i) {
      auto I = std::make_unique<mf::Integral>();
      size_t ls = 0, ss = 0;
      in >> I->type >> I->index >> I->tab_name >> ls >> ss;
      in.get();
      I->tab_src.resize(ls);
      in.read(&I->tab_src[0], static_cast<std::streamsize>(ls));
      I->staged_src.resize(ss);
      if (ss) in.read(&I->staged_src[0], static_cast<std::streamsize>(ss));
      f.ints.push_back(std::move(I));
    }
    if (!in) throw std::runtime_error("truncated description");
    for (int k = 3; k < argc; ++k) {
      const std::string a = argv[k];
      const size_t e = a.find('=');
      f.options[a.substr(0, e)] = std::atoll(a.c_str() + e + 1);
    }
    const std::string src = mf::compile_source(f);
    auto code = mf::rtc_compile(src, "shape_check", mf::rtc_compile_options("gfx950"), "", nullptr);
    std::ofstream(argv[2], std::ios::binary).write(code.data(), static_cast<std::streamsize>(code.size()));
    std::cout << "OK\n";
    return 0;
  } catch (const std::exception& e) {
    std::cout << "FAIL " << e.what() << "\n";
    return 1;
  }
}
