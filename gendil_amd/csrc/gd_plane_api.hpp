// Registry and launch of the plane kernel (gd_plane.hpp): the uniform 3D apply
// for any basis, rule and separable or affine field.
#pragma once

#include <hip/hip_runtime.h>

#include "gd_internal.hpp"

namespace gd {
namespace pl {

constexpr int kVariant = 72;  // gd_plan_set_variant / gd_plan_query_variant code

template <typename T>
struct Args;

template <typename T>
using Launch = int (*)(Args<T>&, const T*, T*, hipStream_t);

struct Entry {
  int N, Q;
  Launch<double> adv64, mass64;
  Launch<float> adv32, mass32;
};

struct List {
  const Entry* e;
  int n;
};

List instances_n2();
List instances_n3();
List instances_n4();
List instances_n5();

// Whether apply() serves this plan.
template <typename T>
bool available(const gd_plan* plan, bool adv, bool mass);

// Whether it is the faster one: always, except that the FP64 advection apply
// with n = 5, q = 6 spills registers and a small mesh cannot hide it (generic
// kernel against this: 216 elements 19 and 24 us with an affine field, 29 and 24
// with one over two coordinates; 1,000 20 and 22, 29 and 21; 1,728 22 and 22, 31
// and 21; 15,625 87 and 77, 122 and 58).
template <typename T>
bool preferred(const gd_plan* plan, bool adv);

// y = mass_coef M x + adv_coef A x; GD_ERR_UNSUPPORTED (nothing launched)
// where no instance serves the plan.
template <typename T>
int apply(const gd_plan* plan, T mass_coef, T adv_coef, const T* x, T* y, hipStream_t s);

}  // namespace pl
}  // namespace gd
