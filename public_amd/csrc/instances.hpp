// Explicit instances of the sweep kernels, in groups that compile side by side:
// each sweeps_*.hip defines one group (INST empty), and the launching unit
// declares them all (INST extern).
#pragma once

#include "adjoint.hpp"
#include "curvilinear.hpp"
#include "sweeps.hpp"

#define INST_SWEEP1(INST, T, Q, DIR, PER, FORM)                                                                  \
  INST template __global__ void cruna::k_sweep1<T, Q, DIR, PER, FORM>(                                            \
      const Q *, T *, T *, cruna::Op<T>, cruna::SweepGeom, cruna::Phys, long, cruna::Metric<T>, cruna::Penal<T>);
#define INST_SWEEP12(INST, T, Q, PER, FORM)                                                                       \
  INST template __global__ void cruna::k_sweep12_z<T, Q, PER, FORM>(                                              \
      const Q *, T *, T *, cruna::Op<T>, cruna::SweepGeom, cruna::Phys, long, cruna::Metric<T>, cruna::Penal<T>);
#define INST_SWEEP2(INST, T, DIR, PER, FORM, FF)                                                                  \
  INST template __global__ void cruna::k_sweep2<T, DIR, PER, FORM, FF>(                                           \
      T *, const T *, cruna::Op<T>, cruna::Op<T>, cruna::SweepGeom, cruna::Phys, long, int, double *, T *, T *,   \
      double, cruna::Metric<T>, const T *, cruna::Penal<T>);
#define INST_CURV1(INST, T, Q, DIR, PER, EV)                                                                      \
  INST template __global__ void cruna::k_curv_sweep1<T, Q, DIR, PER, EV>(                                         \
      const Q *, T *, T *, T *, cruna::Op<T>, cruna::SweepGeom, cruna::Phys, long, cruna::CurvMetric<T>,          \
      cruna::Penal<T>);
#define INST_CURV2(INST, T, DIR, PER, FF, EV)                                                                     \
  INST template __global__ void cruna::k_curv_sweep2<T, DIR, PER, FF, EV>(                                        \
      T *, const T *, const T *, cruna::Op<T>, cruna::Op<T>, cruna::SweepGeom, cruna::Phys, long, int, double *,  \
      T *, T *, double, cruna::CurvMetric<T>, const T *, cruna::Penal<T>);
#define INST_ASWEEP(INST, T, Q, DIR, PER)                                                                         \
  INST template __global__ void cruna::k_asweep<T, Q, DIR, PER>(                                                  \
      const Q *, const double *const *, T *, const double *, cruna::Op<T>, cruna::SweepGeom, double, double,      \
      long, int, double *, T *, T *, double);

// the three forms (Cartesian, tensor-product metric, penalised) of one scheme
#define INST_FORMS1(INST, T, Q, PER)                                                       \
  INST_SWEEP1(INST, T, Q, 0, PER, 0) INST_SWEEP1(INST, T, Q, 1, PER, 0)                    \
  INST_SWEEP12(INST, T, Q, PER, 0)                                                         \
  INST_SWEEP1(INST, T, Q, 0, PER, 1) INST_SWEEP1(INST, T, Q, 1, PER, 1)                    \
  INST_SWEEP12(INST, T, Q, PER, 1)                                                         \
  INST_SWEEP1(INST, T, Q, 0, PER, 2) INST_SWEEP1(INST, T, Q, 1, PER, 2)                    \
  INST_SWEEP12(INST, T, Q, PER, 2)
#define INST_FORMS2(INST, T, PER)                                                          \
  INST_SWEEP2(INST, T, 0, PER, 0, false) INST_SWEEP2(INST, T, 0, PER, 0, true)             \
  INST_SWEEP2(INST, T, 1, PER, 0, false)                                                   \
  INST_SWEEP2(INST, T, 0, PER, 1, false) INST_SWEEP2(INST, T, 0, PER, 1, true)             \
  INST_SWEEP2(INST, T, 1, PER, 1, false)                                                   \
  INST_SWEEP2(INST, T, 0, PER, 2, false) INST_SWEEP2(INST, T, 0, PER, 2, true)             \
  INST_SWEEP2(INST, T, 1, PER, 2, false)
#define INST_CURV_Q(INST, T, Q, PER)                                                       \
  INST_CURV1(INST, T, Q, 0, PER, false) INST_CURV1(INST, T, Q, 0, PER, true)               \
  INST_CURV1(INST, T, Q, 1, PER, false) INST_CURV1(INST, T, Q, 1, PER, true)               \
  INST_CURV1(INST, T, Q, 2, PER, false) INST_CURV1(INST, T, Q, 2, PER, true)
#define INST_CURV_T(INST, T, PER)                                                          \
  INST_CURV2(INST, T, 0, PER, false, false) INST_CURV2(INST, T, 0, PER, false, true)       \
  INST_CURV2(INST, T, 0, PER, true, false) INST_CURV2(INST, T, 0, PER, true, true)         \
  INST_CURV2(INST, T, 1, PER, false, false) INST_CURV2(INST, T, 1, PER, false, true)       \
  INST_CURV2(INST, T, 2, PER, false, false) INST_CURV2(INST, T, 2, PER, false, true)
#define INST_ASWEEPS(INST, T, Q)                                                           \
  INST_ASWEEP(INST, T, Q, 0, true) INST_ASWEEP(INST, T, Q, 0, false)                       \
  INST_ASWEEP(INST, T, Q, 1, true) INST_ASWEEP(INST, T, Q, 1, false)                       \
  INST_ASWEEP(INST, T, Q, 2, true) INST_ASWEEP(INST, T, Q, 2, false)

#define INST_GROUP_PERIODIC64(INST) INST_FORMS1(INST, double, double, true) INST_FORMS2(INST, double, true)
#define INST_GROUP_OPEN64(INST) INST_FORMS1(INST, double, double, false) INST_FORMS2(INST, double, false)
#define INST_GROUP_CURV64(INST) INST_CURV_Q(INST, double, double, true) INST_CURV_T(INST, double, true)
#define INST_GROUP_CURV64O(INST) INST_CURV_Q(INST, double, double, false) INST_CURV_T(INST, double, false)
#define INST_GROUP_FP32(INST)                                                              \
  INST_FORMS1(INST, float, float, true) INST_FORMS1(INST, float, float, false)             \
  INST_FORMS1(INST, float, double, true) INST_FORMS1(INST, float, double, false)
#define INST_GROUP_FP32B(INST)                                                             \
  INST_FORMS2(INST, float, true) INST_FORMS2(INST, float, false)                           \
  INST_CURV_T(INST, float, true) INST_CURV_T(INST, float, false)
#define INST_GROUP_CURV32(INST)                                                            \
  INST_CURV_Q(INST, float, float, true) INST_CURV_Q(INST, float, float, false)             \
  INST_CURV_Q(INST, float, double, true) INST_CURV_Q(INST, float, double, false)
#define INST_GROUP_ADJOINT(INST)                                                           \
  INST_ASWEEPS(INST, double, double) INST_ASWEEPS(INST, float, float) INST_ASWEEPS(INST, float, double)
