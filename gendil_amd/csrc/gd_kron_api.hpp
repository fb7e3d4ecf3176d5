// Registry and launch of the 4D-6D Kronecker kernel (gd_kron.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include "gd_internal.hpp"

namespace gd {
namespace kron {

constexpr int kVariant = 73;  // gd_plan_set_variant / gd_plan_query_variant code

template <typename T>
struct Args;

struct Entry {
  int N;
  int (*f64)(Args<double>&, bool gll, const double*, double*, hipStream_t);
  int (*f32)(Args<float>&, bool gll, const float*, float*, hipStream_t);
};

struct List {
  const Entry* e;
  int n;
};

List instances_d4();
List instances_d5();
List instances_d6();

// Plan-side cache: the terms and their matrices on the device.
struct State;
void destroy_state(State* s);

// Rebuild it for the plan's current coefficients (allocates and copies; called
// by plan creation and every coefficient setter after the device has drained).
int refresh(const gd_plan* plan);

// Whether the kernel serves these coefficients, and whether it is the default
// for them.
bool available(const gd_plan* plan, bool adv, bool mass);
template <typename T>
bool preferred(const gd_plan* plan, bool adv, bool mass);

template <typename T>
int apply(const gd_plan* plan, T mass_coef, T adv_coef, const T* x, T* y, hipStream_t s);

}  // namespace kron
}  // namespace gd
