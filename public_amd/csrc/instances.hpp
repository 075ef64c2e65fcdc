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
#define INST_SWEEP2(INST, T, DIR, PER, FORM, RK, FF)                                                              \
  INST template __global__ void cruna::k_sweep2<T, DIR, PER, FORM, RK, FF>(                                       \
      T *, const T *, cruna::Op<T>, cruna::Op<T>, cruna::SweepGeom, cruna::Phys, long, cruna::RkArgs<T>,          \
      cruna::Metric<T>, const T *, cruna::Penal<T>);
#define INST_CURV1(INST, T, Q, DIR, PER, EV)                                                                      \
  INST template __global__ void cruna::k_curv_sweep1<T, Q, DIR, PER, EV>(                                         \
      const Q *, T *, T *, T *, cruna::Op<T>, cruna::SweepGeom, cruna::Phys, long, cruna::CurvMetric<T>,          \
      cruna::Penal<T>);
#define INST_CURV2(INST, T, DIR, PER, FF, EV, Y)                                                                    \
  INST template __global__ void cruna::k_curv_sweep2<T, DIR, PER, FF, EV, Y>(                                        \
      T *, const T *, const T *, cruna::Op<T>, cruna::Op<T>, cruna::SweepGeom, cruna::Phys, long, int,            \
      cruna::RkArgs<T>, cruna::CurvMetric<T>, const T *, cruna::Penal<T>);
#define INST_ASWEEP(INST, T, Q, DIR, PER, RK)                                                                     \
  INST template __global__ void cruna::k_asweep<T, Q, DIR, PER, RK>(                                              \
      const Q *, const double *const *, T *, const double *, cruna::Op<T>, cruna::SweepGeom, double, double,      \
      long, cruna::RkArgs<T>);

// the three forms (Cartesian, tensor-product metric, penalised) of one scheme
#define INST_FORMS1(INST, T, Q, PER)                                                       \
  INST_SWEEP1(INST, T, Q, 0, PER, 0) INST_SWEEP1(INST, T, Q, 1, PER, 0)                    \
  INST_SWEEP12(INST, T, Q, PER, 0)                                                         \
  INST_SWEEP1(INST, T, Q, 0, PER, 1) INST_SWEEP1(INST, T, Q, 1, PER, 1)                    \
  INST_SWEEP12(INST, T, Q, PER, 1)                                                         \
  INST_SWEEP1(INST, T, Q, 0, PER, 2) INST_SWEEP1(INST, T, Q, 1, PER, 2)                    \
  INST_SWEEP12(INST, T, Q, PER, 2)
// x and y viscous sweeps of one form: every stage update of the x sweep (the
// FP64 forms without an accumulator in FP64 only)
#define INST_FORM2(INST, T, PER, FORM)                                                     \
  INST_SWEEP2(INST, T, 1, PER, FORM, cruna::RK_RHS, false)                                 \
  INST_SWEEP2(INST, T, 0, PER, FORM, cruna::RK_RHS, false)                                 \
  INST_SWEEP2(INST, T, 0, PER, FORM, cruna::RK_FIRST, false)                               \
  INST_SWEEP2(INST, T, 0, PER, FORM, cruna::RK_MID, false)                                 \
  INST_SWEEP2(INST, T, 0, PER, FORM, cruna::RK_LAST, false)
#define INST_FORM2_64(INST, PER, FORM)                                                     \
  INST_FORM2(INST, double, PER, FORM)                                                      \
  INST_SWEEP2(INST, double, 0, PER, FORM, cruna::RK_Y, false)                              \
  INST_SWEEP2(INST, double, 0, PER, FORM, cruna::RK_YLAST, false)                          \
  INST_SWEEP2(INST, double, 0, PER, FORM, cruna::RK_YLAST, true)
#define INST_FORM2_32(INST, PER, FORM)                                                     \
  INST_FORM2(INST, float, PER, FORM)                                                       \
  INST_SWEEP2(INST, float, 0, PER, FORM, cruna::RK_LAST, true)
#define INST_CURV_Q(INST, T, Q, PER)                                                       \
  INST_CURV1(INST, T, Q, 0, PER, false) INST_CURV1(INST, T, Q, 0, PER, true)               \
  INST_CURV1(INST, T, Q, 1, PER, false) INST_CURV1(INST, T, Q, 1, PER, true)               \
  INST_CURV1(INST, T, Q, 2, PER, false) INST_CURV1(INST, T, Q, 2, PER, true)
#define INST_CURV_T(INST, T, PER)                                                          \
  INST_CURV2(INST, T, 0, PER, false, false, false) INST_CURV2(INST, T, 0, PER, false, true, false) \
  INST_CURV2(INST, T, 1, PER, false, false, false) INST_CURV2(INST, T, 1, PER, false, true, false) \
  INST_CURV2(INST, T, 2, PER, false, false, false) INST_CURV2(INST, T, 2, PER, false, true, false)
#define INST_CURV_T64(INST, PER)                                                           \
  INST_CURV_T(INST, double, PER)                                                           \
  INST_CURV2(INST, double, 0, PER, false, false, true) INST_CURV2(INST, double, 0, PER, false, true, true) \
  INST_CURV2(INST, double, 0, PER, true, false, true) INST_CURV2(INST, double, 0, PER, true, true, true)
#define INST_CURV_T32(INST, PER)                                                           \
  INST_CURV_T(INST, float, PER)                                                            \
  INST_CURV2(INST, float, 0, PER, true, false, false) INST_CURV2(INST, float, 0, PER, true, true, false)
#define INST_ASWEEPX(INST, T, Q, PER)                                                      \
  INST_ASWEEP(INST, T, Q, 0, PER, cruna::RK_RHS) INST_ASWEEP(INST, T, Q, 0, PER, cruna::RK_FIRST)
#define INST_ASWEEPX2(INST, T, PER)                                                        \
  INST_ASWEEP(INST, T, T, 0, PER, cruna::RK_MID) INST_ASWEEP(INST, T, T, 0, PER, cruna::RK_LAST)
#define INST_ASWEEPS(INST, T, Q)                                                           \
  INST_ASWEEPX(INST, T, Q, true) INST_ASWEEPX(INST, T, Q, false)                           \
  INST_ASWEEP(INST, T, Q, 1, true, cruna::RK_RHS) INST_ASWEEP(INST, T, Q, 1, false, cruna::RK_RHS) \
  INST_ASWEEP(INST, T, Q, 2, true, cruna::RK_RHS) INST_ASWEEP(INST, T, Q, 2, false, cruna::RK_RHS)

#define INST_GROUP_PERIODIC64(INST)                                                        \
  INST_FORMS1(INST, double, double, true)                                                  \
  INST_FORM2_64(INST, true, 0) INST_FORM2_64(INST, true, 1) INST_FORM2_64(INST, true, 2)
#define INST_GROUP_OPEN64(INST) INST_FORMS1(INST, double, double, false)
#define INST_GROUP_OPEN64B(INST)                                                           \
  INST_FORM2_64(INST, false, 0) INST_FORM2_64(INST, false, 1) INST_FORM2_64(INST, false, 2)
#define INST_GROUP_CURV64(INST) INST_CURV_Q(INST, double, double, true) INST_CURV_T64(INST, true)
#define INST_GROUP_CURV64O(INST) INST_CURV_Q(INST, double, double, false) INST_CURV_T64(INST, false)
#define INST_GROUP_FP32(INST)                                                              \
  INST_FORMS1(INST, float, float, true) INST_FORMS1(INST, float, float, false)             \
  INST_FORMS1(INST, float, double, true) INST_FORMS1(INST, float, double, false)
#define INST_GROUP_FP32B(INST)                                                             \
  INST_FORM2_32(INST, true, 0) INST_FORM2_32(INST, true, 1) INST_FORM2_32(INST, true, 2)    \
  INST_FORM2_32(INST, false, 0) INST_FORM2_32(INST, false, 1) INST_FORM2_32(INST, false, 2) \
  INST_CURV_T32(INST, true) INST_CURV_T32(INST, false)
#define INST_GROUP_CURV32(INST)                                                            \
  INST_CURV_Q(INST, float, float, true) INST_CURV_Q(INST, float, float, false)             \
  INST_CURV_Q(INST, float, double, true) INST_CURV_Q(INST, float, double, false)
#define INST_GROUP_ADJOINT(INST)                                                           \
  INST_ASWEEPS(INST, double, double) INST_ASWEEPS(INST, float, float) INST_ASWEEPS(INST, float, double) \
  INST_ASWEEPX2(INST, double, true) INST_ASWEEPX2(INST, double, false)                     \
  INST_ASWEEPX2(INST, float, true) INST_ASWEEPX2(INST, float, false)                       \
  INST_ASWEEP(INST, double, double, 0, true, cruna::RK_Y) INST_ASWEEP(INST, double, double, 0, false, cruna::RK_Y) \
  INST_ASWEEP(INST, double, double, 0, true, cruna::RK_YLAST)                              \
  INST_ASWEEP(INST, double, double, 0, false, cruna::RK_YLAST)
