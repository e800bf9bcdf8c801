/* Generated by gen_partition.py from fz_atomdata.h (the partition-function
 * programs of atom_database.f90:121-1036).  Do not edit by hand. */
#pragma once

namespace fz {

// REAL(4) AMAX1 of two values, as the programs' AMAX1 opcode
__device__ __forceinline__ double pf_amax1(double x, double y) {
  const float fx = (float)x, fy = (float)y;
  return (double)(fx > fy ? fx : fy);
}

#ifndef PF_DIV
#define PF_DIV(x, y) ((x) / (y))
#define PF_EXP(x) exp(x)
#endif

// One function per element (kept out of line: inlined into one switch the
// 92 bodies are scheduled together and the register demand explodes).
struct PfOut { double u[3], du[3]; };
struct PfVal { double u[3]; };
__device__ __noinline__ PfOut pf_elem_0(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 1.0;
  vUII = 2.0;
  const double t0 = 3.7999998312443495e-05 * vT;
  const double t1 = 1.5099999904632568 + t0;
  const double t2 = (vT > 13000.0) ? 1.0 : 0.0;
  const double t3 = (t2 != 0.0) ? t1 : vUII;
  vUII = t3;
  const double t4 = PF_DIV(3.7999998312443495e-05, vUII);
  const double t5 = (vT > 13000.0) ? 1.0 : 0.0;
  const double t6 = (t5 != 0.0) ? t4 : vDUII;
  vDUII = t6;
  const double t7 = vT * 3.519999935974738e-08;
  const double t8 = -0.0011427999706938863 + t7;
  const double t9 = vT * t8;
  const double t10 = 11.40999984741211 + t9;
  const double t11 = (vT > 16200.0) ? 1.0 : 0.0;
  const double t12 = (t11 != 0.0) ? t10 : vUII;
  vUII = t12;
  const double t13 = 2.0 * vT;
  const double t14 = t13 * 3.519999935974738e-08;
  const double t15 = -0.0011427999706938863 + t14;
  const double t16 = PF_DIV(t15, vUII);
  const double t17 = (vT > 16200.0) ? 1.0 : 0.0;
  const double t18 = (t17 != 0.0) ? t16 : vDUII;
  vDUII = t18;
  vUIII = 1.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_0(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 1.0;
  vUII = 2.0;
  const double t0 = 3.7999998312443495e-05 * vT;
  const double t1 = 1.5099999904632568 + t0;
  const double t2 = (vT > 13000.0) ? 1.0 : 0.0;
  const double t3 = (t2 != 0.0) ? t1 : vUII;
  vUII = t3;
  const double t7 = vT * 3.519999935974738e-08;
  const double t8 = -0.0011427999706938863 + t7;
  const double t9 = vT * t8;
  const double t10 = 11.40999984741211 + t9;
  const double t11 = (vT > 16200.0) ? 1.0 : 0.0;
  const double t12 = (t11 != 0.0) ? t10 : vUII;
  vUII = t12;
  vUIII = 1.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_1(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 1.0;
  const double t0 = vT * 1.609500088761706e-08;
  const double t1 = -0.0009410299826413393 + t0;
  const double t2 = vT * t1;
  const double t3 = 14.800000190734863 + t2;
  const double t4 = (vT > 30000.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vUI;
  vUI = t5;
  const double t6 = 2.0 * vT;
  const double t7 = t6 * 1.609500088761706e-08;
  const double t8 = -0.0009410299826413393 + t7;
  const double t9 = PF_DIV(t8, vUI);
  const double t10 = (vT > 30000.0) ? 1.0 : 0.0;
  const double t11 = (t10 != 0.0) ? t9 : vDUI;
  vDUI = t11;
  vUII = 2.0;
  vUIII = 1.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_1(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 1.0;
  const double t0 = vT * 1.609500088761706e-08;
  const double t1 = -0.0009410299826413393 + t0;
  const double t2 = vT * t1;
  const double t3 = 14.800000190734863 + t2;
  const double t4 = (vT > 30000.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vUI;
  vUI = t5;
  vUII = 2.0;
  vUIII = 1.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_2(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.014081000350415707;
  const double t1 = 0.06892599910497665 - t0;
  const double t2 = vY * t1;
  const double t3 = 2.0810000896453857 - t2;
  vUI = t3;
  const double t4 = 2.0 * vY;
  const double t5 = t4 * 0.014081000350415707;
  const double t6 = -0.06892599910497665 + t5;
  const double t7 = 0.0010000000474974513 * t6;
  const double t8 = PF_DIV(t7, vUI);
  vDUI = t8;
  const double t9 = vT * 8.558600228525393e-08;
  const double t10 = -0.0007329200161620975 + t9;
  const double t11 = vT * t10;
  const double t12 = 3.4863998889923096 + t11;
  const double t13 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t14 = (t13 != 0.0) ? t12 : vUI;
  vUI = t14;
  const double t15 = 2.0 * vT;
  const double t16 = t15 * 8.558600228525393e-08;
  const double t17 = -0.0007329200161620975 + t16;
  const double t18 = PF_DIV(t17, vUI);
  const double t19 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t20 = (t19 != 0.0) ? t18 : vDUI;
  vDUI = t20;
  vUII = 1.0;
  vUIII = 2.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_2(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.014081000350415707;
  const double t1 = 0.06892599910497665 - t0;
  const double t2 = vY * t1;
  const double t3 = 2.0810000896453857 - t2;
  vUI = t3;
  const double t9 = vT * 8.558600228525393e-08;
  const double t10 = -0.0007329200161620975 + t9;
  const double t11 = vT * t10;
  const double t12 = 3.4863998889923096 + t11;
  const double t13 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t14 = (t13 != 0.0) ? t12 : vUI;
  vUI = t14;
  vUII = 1.0;
  vUIII = 2.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_3(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 7.031999848550186e-05 * vT;
  const double t1 = 0.6309999823570251 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(7.031999848550186e-05, vUI);
  const double t4 = (vUI != 1.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  vUII = 2.0;
  vUIII = 1.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_3(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 7.031999848550186e-05 * vT;
  const double t1 = 0.6309999823570251 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  vUII = 2.0;
  vUIII = 1.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_4(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.010437999852001667 * vY;
  const double t1 = 5.935100078582764 + t0;
  vUI = t1;
  const double t2 = PF_DIV(1.043800057232147e-05, vUI);
  vDUI = t2;
  vUII = 1.0;
  vUIII = 2.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_4(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.010437999852001667 * vY;
  const double t1 = 5.935100078582764 + t0;
  vUI = t1;
  vUII = 1.0;
  vUIII = 2.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_5(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.00039090999052859843 * vY;
  const double t1 = 0.017628999426960945 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.02048500068485737 + t2;
  const double t4 = vY * t3;
  const double t5 = 8.69849967956543 + t4;
  vUI = t5;
  const double t6 = 2.0 * vY;
  const double t7 = t6 * 0.017628999426960945;
  const double t8 = 0.02048500068485737 + t7;
  const double t9 = 3.0 * vY;
  const double t10 = t9 * vY;
  const double t11 = t10 * 0.00039090999052859843;
  const double t12 = t8 - t11;
  const double t13 = PF_DIV(t12, vUI);
  const double t14 = 0.0010000000474974513 * t13;
  vDUI = t14;
  const double t15 = vT * 9.08439972135966e-08;
  const double t16 = -0.0013906999956816435 + t15;
  const double t17 = vT * t16;
  const double t18 = 13.970000267028809 + t17;
  const double t19 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t20 = (t19 != 0.0) ? t18 : vUI;
  vUI = t20;
  const double t21 = 2.0 * vT;
  const double t22 = t21 * 9.08439972135966e-08;
  const double t23 = -0.0013906999956816435 + t22;
  const double t24 = PF_DIV(t23, vUI);
  const double t25 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t26 = (t25 != 0.0) ? t24 : vDUI;
  vDUI = t26;
  const double t27 = 1.6833000699989498e-05 * vT;
  const double t28 = 5.8379998207092285 + t27;
  vUII = t28;
  const double t29 = PF_DIV(1.6833000699989498e-05, vUII);
  vDUII = t29;
  const double t30 = vT * 2.0861000038507882e-08;
  const double t31 = -0.0006934700068086386 + t30;
  const double t32 = vT * t31;
  const double t33 = 10.98900032043457 + t32;
  const double t34 = (vT > 24000.0) ? 1.0 : 0.0;
  const double t35 = (t34 != 0.0) ? t33 : vUII;
  vUII = t35;
  const double t36 = 2.0 * vT;
  const double t37 = t36 * 2.0861000038507882e-08;
  const double t38 = -0.0006934700068086386 + t37;
  const double t39 = PF_DIV(t38, vUII);
  const double t40 = (vT > 24000.0) ? 1.0 : 0.0;
  const double t41 = (t40 != 0.0) ? t39 : vDUII;
  vDUII = t41;
  vUIII = 1.0;
  const double t42 = 7.999999797903001e-05 * vT;
  const double t43 = -0.5550000071525574 + t42;
  const double t44 = (vT > 19500.0) ? 1.0 : 0.0;
  const double t45 = (t44 != 0.0) ? t43 : vUIII;
  vUIII = t45;
  const double t46 = PF_DIV(7.999999797903001e-05, vUIII);
  const double t47 = (vT > 19500.0) ? 1.0 : 0.0;
  const double t48 = (t47 != 0.0) ? t46 : vDUIII;
  vDUIII = t48;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_5(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.00039090999052859843 * vY;
  const double t1 = 0.017628999426960945 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.02048500068485737 + t2;
  const double t4 = vY * t3;
  const double t5 = 8.69849967956543 + t4;
  vUI = t5;
  const double t15 = vT * 9.08439972135966e-08;
  const double t16 = -0.0013906999956816435 + t15;
  const double t17 = vT * t16;
  const double t18 = 13.970000267028809 + t17;
  const double t19 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t20 = (t19 != 0.0) ? t18 : vUI;
  vUI = t20;
  const double t27 = 1.6833000699989498e-05 * vT;
  const double t28 = 5.8379998207092285 + t27;
  vUII = t28;
  const double t30 = vT * 2.0861000038507882e-08;
  const double t31 = -0.0006934700068086386 + t30;
  const double t32 = vT * t31;
  const double t33 = 10.98900032043457 + t32;
  const double t34 = (vT > 24000.0) ? 1.0 : 0.0;
  const double t35 = (t34 != 0.0) ? t33 : vUII;
  vUII = t35;
  vUIII = 1.0;
  const double t42 = 7.999999797903001e-05 * vT;
  const double t43 = -0.5550000071525574 + t42;
  const double t44 = (vT > 19500.0) ? 1.0 : 0.0;
  const double t45 = (t44 != 0.0) ? t43 : vUIII;
  vUIII = t45;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_6(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.001713800011202693;
  const double t1 = 0.010147999972105026 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.017490999773144722 - t2;
  const double t4 = vY * t3;
  const double t5 = 3.9914000034332275 + t4;
  vUI = t5;
  const double t6 = 2.0 * vY;
  const double t7 = t6 * 0.010147999972105026;
  const double t8 = 0.017490999773144722 - t7;
  const double t9 = 3.0 * vY;
  const double t10 = t9 * vY;
  const double t11 = t10 * 0.001713800011202693;
  const double t12 = t8 + t11;
  const double t13 = PF_DIV(t12, vUI);
  const double t14 = 0.0010000000474974513 * t13;
  vDUI = t14;
  const double t15 = 0.00025400001322850585 * vT;
  const double t16 = 2.1710000038146973 + t15;
  const double t17 = (vT > 8800.0) ? 1.0 : 0.0;
  const double t18 = (t17 != 0.0) ? t16 : vUI;
  vUI = t18;
  const double t19 = PF_DIV(0.00025400001322850585, vUI);
  const double t20 = (vT > 8800.0) ? 1.0 : 0.0;
  const double t21 = (t20 != 0.0) ? t19 : vDUI;
  vDUI = t21;
  const double t22 = vT * 8.632999737301361e-08;
  const double t23 = -0.0017139000119641423 + t22;
  const double t24 = vT * t23;
  const double t25 = 11.395999908447266 + t24;
  const double t26 = (vT > 18000.0) ? 1.0 : 0.0;
  const double t27 = (t26 != 0.0) ? t25 : vUI;
  vUI = t27;
  const double t28 = 2.0 * vT;
  const double t29 = t28 * 8.632999737301361e-08;
  const double t30 = -0.0017139000119641423 + t29;
  const double t31 = PF_DIV(t30, vUI);
  const double t32 = (vT > 18000.0) ? 1.0 : 0.0;
  const double t33 = (t32 != 0.0) ? t31 : vDUI;
  vDUI = t33;
  const double t34 = 0.00014200000441633165 * vT;
  const double t35 = 8.0600004196167 + t34;
  vUII = t35;
  const double t36 = PF_DIV(0.00014200000441633165, vUII);
  vDUII = t36;
  const double t37 = vT * 4.4612001204313856e-08;
  const double t38 = -0.0018930999794974923 + t37;
  const double t39 = vT * t38;
  const double t40 = 26.792999267578125 + t39;
  const double t41 = (vT > 33000.0) ? 1.0 : 0.0;
  const double t42 = (t41 != 0.0) ? t40 : vUII;
  vUII = t42;
  const double t43 = 2.0 * vT;
  const double t44 = t43 * 4.4612001204313856e-08;
  const double t45 = -0.0018930999794974923 + t44;
  const double t46 = PF_DIV(t45, vUII);
  const double t47 = (vT > 33000.0) ? 1.0 : 0.0;
  const double t48 = (t47 != 0.0) ? t46 : vDUII;
  vDUII = t48;
  const double t49 = vT * 1.8228000220332774e-09;
  const double t50 = -2.6650999643607065e-05 + t49;
  const double t51 = vT * t50;
  const double t52 = 5.983500003814697 + t51;
  vUIII = t52;
  const double t53 = 2.0 * vT;
  const double t54 = t53 * 1.8228000220332774e-09;
  const double t55 = -2.6650999643607065e-05 + t54;
  const double t56 = PF_DIV(t55, vUIII);
  vDUIII = t56;
  const double t57 = (vT < 7310.5) ? 1.0 : 0.0;
  const double t58 = (t57 != 0.0) ? 5.889999866485596 : vUIII;
  vUIII = t58;
  const double t59 = (vT < 7310.5) ? 1.0 : 0.0;
  const double t60 = (t59 != 0.0) ? 0.0 : vDUIII;
  vDUIII = t60;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_6(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.001713800011202693;
  const double t1 = 0.010147999972105026 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.017490999773144722 - t2;
  const double t4 = vY * t3;
  const double t5 = 3.9914000034332275 + t4;
  vUI = t5;
  const double t15 = 0.00025400001322850585 * vT;
  const double t16 = 2.1710000038146973 + t15;
  const double t17 = (vT > 8800.0) ? 1.0 : 0.0;
  const double t18 = (t17 != 0.0) ? t16 : vUI;
  vUI = t18;
  const double t22 = vT * 8.632999737301361e-08;
  const double t23 = -0.0017139000119641423 + t22;
  const double t24 = vT * t23;
  const double t25 = 11.395999908447266 + t24;
  const double t26 = (vT > 18000.0) ? 1.0 : 0.0;
  const double t27 = (t26 != 0.0) ? t25 : vUI;
  vUI = t27;
  const double t34 = 0.00014200000441633165 * vT;
  const double t35 = 8.0600004196167 + t34;
  vUII = t35;
  const double t37 = vT * 4.4612001204313856e-08;
  const double t38 = -0.0018930999794974923 + t37;
  const double t39 = vT * t38;
  const double t40 = 26.792999267578125 + t39;
  const double t41 = (vT > 33000.0) ? 1.0 : 0.0;
  const double t42 = (t41 != 0.0) ? t40 : vUII;
  vUII = t42;
  const double t49 = vT * 1.8228000220332774e-09;
  const double t50 = -2.6650999643607065e-05 + t49;
  const double t51 = vT * t50;
  const double t52 = 5.983500003814697 + t51;
  vUIII = t52;
  const double t57 = (vT < 7310.5) ? 1.0 : 0.0;
  const double t58 = (t57 != 0.0) ? 5.889999866485596 : vUIII;
  vUIII = t58;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_7(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.00011000000085914508 * vT;
  const double t1 = 8.289999961853027 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.00011000000085914508, vUI);
  vDUI = t2;
  const double t3 = vT * 1.657000012755816e-07;
  const double t4 = -0.0060189999639987946 + t3;
  const double t5 = vT * t4;
  const double t6 = 66.80999755859375 + t5;
  const double t7 = (vT > 19000.0) ? 1.0 : 0.0;
  const double t8 = (t7 != 0.0) ? t6 : vUI;
  vUI = t8;
  const double t9 = 2.0 * vT;
  const double t10 = t9 * 1.657000012755816e-07;
  const double t11 = -0.0060189999639987946 + t10;
  const double t12 = PF_DIV(t11, vUI);
  const double t13 = (vT > 19000.0) ? 1.0 : 0.0;
  const double t14 = (t13 != 0.0) ? t12 : vDUI;
  vDUI = t14;
  const double t15 = 7.999999797903001e-05 * vT;
  const double t16 = 3.509999990463257 + t15;
  const double t17 = (4.0 > t16) ? 4.0 : t16;
  vUII = t17;
  const double t18 = PF_DIV(7.999999797903001e-05, vUII);
  const double t19 = (vUII != 4.0) ? 1.0 : 0.0;
  const double t20 = (t19 != 0.0) ? t18 : vDUII;
  vDUII = t20;
  const double t21 = vT * 6.88499994794256e-08;
  const double t22 = -0.004215999972075224 + t21;
  const double t23 = vT * t22;
  const double t24 = 68.69999694824219 + t23;
  const double t25 = (vT > 36400.0) ? 1.0 : 0.0;
  const double t26 = (t25 != 0.0) ? t24 : vUII;
  vUII = t26;
  const double t27 = 2.0 * vT;
  const double t28 = t27 * 6.88499994794256e-08;
  const double t29 = -0.004215999972075224 + t28;
  const double t30 = PF_DIV(t29, vUII);
  const double t31 = (vT > 36400.0) ? 1.0 : 0.0;
  const double t32 = (t31 != 0.0) ? t30 : vDUII;
  vDUII = t32;
  const double t33 = 0.00011347999679856002 * vT;
  const double t34 = 7.864999771118164 + t33;
  vUIII = t34;
  const double t35 = PF_DIV(0.00011347999679856002, vUIII);
  vDUIII = t35;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_7(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.00011000000085914508 * vT;
  const double t1 = 8.289999961853027 + t0;
  vUI = t1;
  const double t3 = vT * 1.657000012755816e-07;
  const double t4 = -0.0060189999639987946 + t3;
  const double t5 = vT * t4;
  const double t6 = 66.80999755859375 + t5;
  const double t7 = (vT > 19000.0) ? 1.0 : 0.0;
  const double t8 = (t7 != 0.0) ? t6 : vUI;
  vUI = t8;
  const double t15 = 7.999999797903001e-05 * vT;
  const double t16 = 3.509999990463257 + t15;
  const double t17 = (4.0 > t16) ? 4.0 : t16;
  vUII = t17;
  const double t21 = vT * 6.88499994794256e-08;
  const double t22 = -0.004215999972075224 + t21;
  const double t23 = vT * t22;
  const double t24 = 68.69999694824219 + t23;
  const double t25 = (vT > 36400.0) ? 1.0 : 0.0;
  const double t26 = (t25 != 0.0) ? t24 : vUII;
  vUII = t26;
  const double t33 = 0.00011347999679856002 * vT;
  const double t34 = 7.864999771118164 + t33;
  vUIII = t34;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_8(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0013035000301897526 * vY;
  const double t1 = 0.026770999655127525 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.2088399976491928 + t2;
  const double t4 = vY * t3;
  const double t5 = 0.7768300175666809 + t4;
  const double t6 = vY * t5;
  const double t7 = 4.583199977874756 + t6;
  vUI = t7;
  const double t8 = 2.0 * vY;
  const double t9 = t8 * 0.2088399976491928;
  const double t10 = 0.7768300175666809 - t9;
  const double t11 = 3.0 * vY;
  const double t12 = t11 * vY;
  const double t13 = t12 * 0.026770999655127525;
  const double t14 = t10 + t13;
  const double t15 = 4.0 * vY;
  const double t16 = t15 * vY;
  const double t17 = t16 * vY;
  const double t18 = t17 * 0.0013035000301897526;
  const double t19 = t14 - t18;
  vDUI = t19;
  const double t20 = PF_DIV(vDUI, vUI);
  const double t21 = 0.0010000000474974513 * t20;
  vDUI = t21;
  const double t22 = (vT > 8750.0) ? 1.0 : 0.0;
  const double t23 = (t22 != 0.0) ? 5.900000095367432 : vUI;
  vUI = t23;
  const double t24 = (vT > 8750.0) ? 1.0 : 0.0;
  const double t25 = (t24 != 0.0) ? 0.0 : vDUI;
  vDUI = t25;
  const double t26 = vT * 2.3120000136600538e-08;
  const double t27 = -0.0009228999842889607 + t26;
  const double t28 = vT * t27;
  const double t29 = 15.15999984741211 + t28;
  const double t30 = (vT > 20000.0) ? 1.0 : 0.0;
  const double t31 = (t30 != 0.0) ? t29 : vUI;
  vUI = t31;
  const double t32 = 2.0 * vT;
  const double t33 = t32 * 2.3120000136600538e-08;
  const double t34 = -0.0009228999842889607 + t33;
  const double t35 = PF_DIV(t34, vUI);
  const double t36 = (vT > 20000.0) ? 1.0 : 0.0;
  const double t37 = (t36 != 0.0) ? t35 : vDUI;
  vDUI = t37;
  const double t38 = 8.900000102585182e-05 * vT;
  const double t39 = 8.149999618530273 + t38;
  vUII = t39;
  const double t40 = PF_DIV(8.900000102585182e-05, vUII);
  vDUII = t40;
  const double t41 = 0.00013800000306218863 * vT;
  const double t42 = 2.315000057220459 + t41;
  vUIII = t42;
  const double t43 = PF_DIV(0.00013800000306218863, vUIII);
  vDUIII = t43;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_8(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0013035000301897526 * vY;
  const double t1 = 0.026770999655127525 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.2088399976491928 + t2;
  const double t4 = vY * t3;
  const double t5 = 0.7768300175666809 + t4;
  const double t6 = vY * t5;
  const double t7 = 4.583199977874756 + t6;
  vUI = t7;
  const double t22 = (vT > 8750.0) ? 1.0 : 0.0;
  const double t23 = (t22 != 0.0) ? 5.900000095367432 : vUI;
  vUI = t23;
  const double t26 = vT * 2.3120000136600538e-08;
  const double t27 = -0.0009228999842889607 + t26;
  const double t28 = vT * t27;
  const double t29 = 15.15999984741211 + t28;
  const double t30 = (vT > 20000.0) ? 1.0 : 0.0;
  const double t31 = (t30 != 0.0) ? t29 : vUI;
  vUI = t31;
  const double t38 = 8.900000102585182e-05 * vT;
  const double t39 = 8.149999618530273 + t38;
  vUII = t39;
  const double t41 = 0.00013800000306218863 * vT;
  const double t42 = 2.315000057220459 + t41;
  vUIII = t42;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_9(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 1.0;
  const double t0 = vT * 4.3589999165760673e-08;
  const double t1 = -0.002113000024110079 + t0;
  const double t2 = vT * t1;
  const double t3 = 26.299999237060547 + t2;
  const double t4 = (vT > 26900.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vUI;
  vUI = t5;
  const double t6 = 2.0 * vT;
  const double t7 = t6 * 4.3589999165760673e-08;
  const double t8 = -0.002113000024110079 + t7;
  const double t9 = PF_DIV(t8, vUI);
  const double t10 = (vT > 26900.0) ? 1.0 : 0.0;
  const double t11 = (t10 != 0.0) ? t9 : vDUI;
  vDUI = t11;
  const double t12 = 3.9999998989515007e-05 * vT;
  const double t13 = 5.400000095367432 + t12;
  vUII = t13;
  const double t14 = PF_DIV(3.9999998989515007e-05, vUII);
  vDUII = t14;
  const double t15 = 7.95599989942275e-05 * vT;
  const double t16 = 7.9730000495910645 + t15;
  vUIII = t16;
  const double t17 = PF_DIV(7.95599989942275e-05, vUIII);
  vDUIII = t17;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_9(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 1.0;
  const double t0 = vT * 4.3589999165760673e-08;
  const double t1 = -0.002113000024110079 + t0;
  const double t2 = vT * t1;
  const double t3 = 26.299999237060547 + t2;
  const double t4 = (vT > 26900.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vUI;
  vUI = t5;
  const double t12 = 3.9999998989515007e-05 * vT;
  const double t13 = 5.400000095367432 + t12;
  vUII = t13;
  const double t15 = 7.95599989942275e-05 * vT;
  const double t16 = 7.9730000495910645 + t15;
  vUIII = t16;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_10(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 9.300000237999484e-05 * vT;
  const double t1 = 1.7200000286102295 + t0;
  const double t2 = (2.0 > t1) ? 2.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(9.300000237999484e-05, vUI);
  const double t4 = (vUI != 2.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  const double t6 = 0.0005660000024363399 * vT;
  const double t7 = -0.8299999833106995 + t6;
  const double t8 = (vT > 5400.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t10 = PF_DIV(0.0005660000024363399, vUI);
  const double t11 = (vT > 5400.0) ? 1.0 : 0.0;
  const double t12 = (t11 != 0.0) ? t10 : vDUI;
  vDUI = t12;
  const double t13 = vT * 1.3861000525139389e-07;
  const double t14 = -0.001241500023752451 + t13;
  const double t15 = vT * t14;
  const double t16 = 4.55679988861084 + t15;
  const double t17 = (vT > 8500.0) ? 1.0 : 0.0;
  const double t18 = (t17 != 0.0) ? t16 : vUI;
  vUI = t18;
  const double t19 = 2.0 * vT;
  const double t20 = t19 * 1.3861000525139389e-07;
  const double t21 = -0.001241500023752451 + t20;
  const double t22 = PF_DIV(t21, vUI);
  const double t23 = (vT > 8500.0) ? 1.0 : 0.0;
  const double t24 = (t23 != 0.0) ? t22 : vDUI;
  vDUI = t24;
  vUII = 1.0;
  const double t25 = 5.689999852620531e-06 * vT;
  const double t26 = 5.690000057220459 + t25;
  vUIII = t26;
  const double t27 = PF_DIV(5.689999852620531e-06, vUIII);
  vDUIII = t27;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_10(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 9.300000237999484e-05 * vT;
  const double t1 = 1.7200000286102295 + t0;
  const double t2 = (2.0 > t1) ? 2.0 : t1;
  vUI = t2;
  const double t6 = 0.0005660000024363399 * vT;
  const double t7 = -0.8299999833106995 + t6;
  const double t8 = (vT > 5400.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t13 = vT * 1.3861000525139389e-07;
  const double t14 = -0.001241500023752451 + t13;
  const double t15 = vT * t14;
  const double t16 = 4.55679988861084 + t15;
  const double t17 = (vT > 8500.0) ? 1.0 : 0.0;
  const double t18 = (t17 != 0.0) ? t16 : vUI;
  vUI = t18;
  vUII = 1.0;
  const double t25 = 5.689999852620531e-06 * vT;
  const double t26 = 5.690000057220459 + t25;
  vUIII = t26;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_11(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.7841309905052185 * vX;
  const double t1 = 2.393894910812378 + t0;
  const double t2 = vX * t1;
  const double t3 = 2.8891758918762207 + t2;
  const double t4 = vX * t3;
  const double t5 = 6.1731719970703125 + t4;
  const double t6 = vX * t5;
  const double t7 = -4.027262210845947 - t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 1.0 + t8;
  vUI = t9;
  const double t10 = 4.0 * vX;
  const double t11 = t10 * 0.7841309905052185;
  const double t12 = 7.181684494018555 + t11;
  const double t13 = vX * t12;
  const double t14 = 5.778351783752441 + t13;
  const double t15 = vX * t14;
  const double t16 = 6.1731719970703125 + t15;
  const double t17 = vDX * t16;
  const double t18 = -t17;
  vDUI = t18;
  const double t19 = vUI - 1.0;
  const double t20 = vDUI * t19;
  const double t21 = PF_DIV(t20, vUI);
  vDUI = t21;
  const double t22 = vT * 7.453100181464833e-08;
  const double t23 = -0.0007890900014899671 + t22;
  const double t24 = vT * t23;
  const double t25 = 2.756999969482422 + t24;
  const double t26 = (vT > 8000.0) ? 1.0 : 0.0;
  const double t27 = (t26 != 0.0) ? t25 : vUI;
  vUI = t27;
  const double t28 = 2.0 * vT;
  const double t29 = t28 * 7.453100181464833e-08;
  const double t30 = -0.0007890900014899671 + t29;
  const double t31 = PF_DIV(t30, vUI);
  const double t32 = (vT > 8000.0) ? 1.0 : 0.0;
  const double t33 = (t32 != 0.0) ? t31 : vDUI;
  vDUI = t33;
  const double t34 = 0.21241700649261475 * vX;
  const double t35 = 1.9660969972610474 + t34;
  const double t36 = vX * t35;
  const double t37 = 7.600677967071533 + t36;
  const double t38 = vX * t37;
  const double t39 = -7.721171855926514 - t38;
  const double t40 = PF_EXP(t39);
  const double t41 = 2.0 + t40;
  vUII = t41;
  const double t42 = 3.0 * vX;
  const double t43 = t42 * 0.21241700649261475;
  const double t44 = 3.9321939945220947 + t43;
  const double t45 = vX * t44;
  const double t46 = 7.060067653656006 + t45;
  const double t47 = vDX * t46;
  const double t48 = -t47;
  vDUII = t48;
  const double t49 = vUII - 2.0;
  const double t50 = vDUII * t49;
  const double t51 = PF_DIV(t50, vUII);
  vDUII = t51;
  const double t52 = vT * 4.784099871812941e-08;
  const double t53 = -0.0010816999711096287 + t52;
  const double t54 = vT * t53;
  const double t55 = 7.104100227355957 + t54;
  const double t56 = (vT > 20000.0) ? 1.0 : 0.0;
  const double t57 = (t56 != 0.0) ? t55 : vUII;
  vUII = t57;
  const double t58 = 2.0 * vT;
  const double t59 = t58 * 4.784099871812941e-08;
  const double t60 = -0.0010816999711096287 + t59;
  const double t61 = PF_DIV(t60, vUII);
  const double t62 = (vT > 20000.0) ? 1.0 : 0.0;
  const double t63 = (t62 != 0.0) ? t61 : vDUII;
  vDUII = t63;
  vUIII = 1.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_11(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.7841309905052185 * vX;
  const double t1 = 2.393894910812378 + t0;
  const double t2 = vX * t1;
  const double t3 = 2.8891758918762207 + t2;
  const double t4 = vX * t3;
  const double t5 = 6.1731719970703125 + t4;
  const double t6 = vX * t5;
  const double t7 = -4.027262210845947 - t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 1.0 + t8;
  vUI = t9;
  const double t22 = vT * 7.453100181464833e-08;
  const double t23 = -0.0007890900014899671 + t22;
  const double t24 = vT * t23;
  const double t25 = 2.756999969482422 + t24;
  const double t26 = (vT > 8000.0) ? 1.0 : 0.0;
  const double t27 = (t26 != 0.0) ? t25 : vUI;
  vUI = t27;
  const double t34 = 0.21241700649261475 * vX;
  const double t35 = 1.9660969972610474 + t34;
  const double t36 = vX * t35;
  const double t37 = 7.600677967071533 + t36;
  const double t38 = vX * t37;
  const double t39 = -7.721171855926514 - t38;
  const double t40 = PF_EXP(t39);
  const double t41 = 2.0 + t40;
  vUII = t41;
  const double t52 = vT * 4.784099871812941e-08;
  const double t53 = -0.0010816999711096287 + t52;
  const double t54 = vT * t53;
  const double t55 = 7.104100227355957 + t54;
  const double t56 = (vT > 20000.0) ? 1.0 : 0.0;
  const double t57 = (t56 != 0.0) ? t55 : vUII;
  vUII = t57;
  vUIII = 1.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_12(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.0030199000611901283;
  const double t1 = 0.04752900078892708 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.278329998254776 - t2;
  const double t4 = vY * t3;
  const double t5 = 5.295499801635742 + t4;
  vUI = t5;
  const double t6 = 3.0 * vY;
  const double t7 = t6 * 0.0030199000611901283;
  const double t8 = 0.09505800157785416 - t7;
  const double t9 = vY * t8;
  const double t10 = 0.278329998254776 - t9;
  const double t11 = 0.0010000000474974513 * t10;
  const double t12 = PF_DIV(t11, vUI);
  vDUI = t12;
  const double t13 = 3.2449999707750976e-05 * vT;
  const double t14 = 0.7250000238418579 + t13;
  const double t15 = (1.0 > t14) ? 1.0 : t14;
  vUII = t15;
  const double t16 = PF_DIV(3.2449999707750976e-05, vUII);
  const double t17 = (vUII != 1.0) ? 1.0 : 0.0;
  const double t18 = (t17 != 0.0) ? t16 : vDUII;
  vDUII = t18;
  const double t19 = vT * 1.4850000695787458e-07;
  const double t20 = -0.005987000185996294 + t19;
  const double t21 = vT * t20;
  const double t22 = 61.060001373291016 + t21;
  const double t23 = (vT > 22400.0) ? 1.0 : 0.0;
  const double t24 = (t23 != 0.0) ? t22 : vUII;
  vUII = t24;
  const double t25 = 2.0 * vT;
  const double t26 = t25 * 1.4850000695787458e-07;
  const double t27 = -0.005987000185996294 + t26;
  const double t28 = PF_DIV(t27, vUII);
  const double t29 = (vT > 22400.0) ? 1.0 : 0.0;
  const double t30 = (t29 != 0.0) ? t28 : vDUII;
  vDUII = t30;
  const double t31 = 3.4300001061637886e-06 * vT;
  const double t32 = 1.9759999513626099 + t31;
  const double t33 = (2.0 > t32) ? 2.0 : t32;
  vUIII = t33;
  const double t34 = PF_DIV(3.4300001061637886e-06, vUIII);
  const double t35 = (vUIII != 2.0) ? 1.0 : 0.0;
  const double t36 = (t35 != 0.0) ? t34 : vDUIII;
  vDUIII = t36;
  const double t37 = vT * 4.38200009611478e-09;
  const double t38 = -0.00015900000289548188 + t37;
  const double t39 = vT * t38;
  const double t40 = 3.5220000743865967 + t39;
  const double t41 = (vT > 18140.0) ? 1.0 : 0.0;
  const double t42 = (t41 != 0.0) ? t40 : vUIII;
  vUIII = t42;
  const double t43 = 2.0 * vT;
  const double t44 = t43 * 4.38200009611478e-09;
  const double t45 = -0.00015900000289548188 + t44;
  const double t46 = PF_DIV(t45, vUIII);
  const double t47 = (vT > 18140.0) ? 1.0 : 0.0;
  const double t48 = (t47 != 0.0) ? t46 : vDUIII;
  vDUIII = t48;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_12(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.0030199000611901283;
  const double t1 = 0.04752900078892708 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.278329998254776 - t2;
  const double t4 = vY * t3;
  const double t5 = 5.295499801635742 + t4;
  vUI = t5;
  const double t13 = 3.2449999707750976e-05 * vT;
  const double t14 = 0.7250000238418579 + t13;
  const double t15 = (1.0 > t14) ? 1.0 : t14;
  vUII = t15;
  const double t19 = vT * 1.4850000695787458e-07;
  const double t20 = -0.005987000185996294 + t19;
  const double t21 = vT * t20;
  const double t22 = 61.060001373291016 + t21;
  const double t23 = (vT > 22400.0) ? 1.0 : 0.0;
  const double t24 = (t23 != 0.0) ? t22 : vUII;
  vUII = t24;
  const double t31 = 3.4300001061637886e-06 * vT;
  const double t32 = 1.9759999513626099 + t31;
  const double t33 = (2.0 > t32) ? 2.0 : t32;
  vUIII = t33;
  const double t37 = vT * 4.38200009611478e-09;
  const double t38 = -0.00015900000289548188 + t37;
  const double t39 = vT * t38;
  const double t40 = 3.5220000743865967 + t39;
  const double t41 = (vT > 18140.0) ? 1.0 : 0.0;
  const double t42 = (t41 != 0.0) ? t40 : vUIII;
  vUIII = t42;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_13(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0006201299838721752 * vY;
  const double t1 = 0.013109000399708748 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.11621999740600586 + t2;
  const double t4 = vY * t3;
  const double t5 = 0.8631899952888489 + t4;
  const double t6 = vY * t5;
  const double t7 = 6.786799907684326 + t6;
  vUI = t7;
  const double t8 = 4.0 * vY;
  const double t9 = t8 * 0.0006201299838721752;
  const double t10 = 0.03932700306177139 - t9;
  const double t11 = vY * t10;
  const double t12 = -0.23243999481201172 + t11;
  const double t13 = vY * t12;
  const double t14 = 0.8631899952888489 + t13;
  const double t15 = 0.0010000000474974513 * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = vT * 7.28200006960833e-07;
  const double t18 = -0.014650000259280205 + t17;
  const double t19 = vT * t18;
  const double t20 = 86.01000213623047 + t19;
  const double t21 = (vT > 10400.0) ? 1.0 : 0.0;
  const double t22 = (t21 != 0.0) ? t20 : vUI;
  vUI = t22;
  const double t23 = 2.0 * vT;
  const double t24 = t23 * 7.28200006960833e-07;
  const double t25 = -0.014650000259280205 + t24;
  const double t26 = PF_DIV(t25, vUI);
  const double t27 = (vT > 10400.0) ? 1.0 : 0.0;
  const double t28 = (t27 != 0.0) ? t26 : vDUI;
  vDUI = t28;
  const double t29 = 3.9999998989515007e-05 * vT;
  const double t30 = 5.46999979019165 + t29;
  vUII = t30;
  const double t31 = PF_DIV(3.9999998989515007e-05, vUII);
  vDUII = t31;
  const double t32 = vT * 6.188000156726048e-08;
  const double t33 = -0.002219999907538295 + t32;
  const double t34 = vT * t33;
  const double t35 = 26.440000534057617 + t34;
  const double t36 = (vT > 18000.0) ? 1.0 : 0.0;
  const double t37 = (t36 != 0.0) ? t35 : vUII;
  vUII = t37;
  const double t38 = 2.0 * vT;
  const double t39 = t38 * 6.188000156726048e-08;
  const double t40 = -0.002219999907538295 + t39;
  const double t41 = PF_DIV(t40, vUII);
  const double t42 = (vT > 18000.0) ? 1.0 : 0.0;
  const double t43 = (t42 != 0.0) ? t41 : vDUII;
  vDUII = t43;
  const double t44 = 1.1000000085914508e-05 * vT;
  const double t45 = 0.9110000133514404 + t44;
  const double t46 = (1.0 > t45) ? 1.0 : t45;
  vUIII = t46;
  const double t47 = PF_DIV(1.1000000085914508e-05, vUIII);
  const double t48 = (vUIII != 1.0) ? 1.0 : 0.0;
  const double t49 = (t48 != 0.0) ? t47 : vDUIII;
  vDUIII = t49;
  const double t50 = vT * 2.616999950078025e-08;
  const double t51 = -0.001408000010997057 + t50;
  const double t52 = vT * t51;
  const double t53 = 19.139999389648438 + t52;
  const double t54 = (vT > 33300.0) ? 1.0 : 0.0;
  const double t55 = (t54 != 0.0) ? t53 : vUIII;
  vUIII = t55;
  const double t56 = 2.0 * vT;
  const double t57 = t56 * 2.616999950078025e-08;
  const double t58 = -0.001408000010997057 + t57;
  const double t59 = PF_DIV(t58, vUIII);
  const double t60 = (vT > 33300.0) ? 1.0 : 0.0;
  const double t61 = (t60 != 0.0) ? t59 : vDUIII;
  vDUIII = t61;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_13(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0006201299838721752 * vY;
  const double t1 = 0.013109000399708748 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.11621999740600586 + t2;
  const double t4 = vY * t3;
  const double t5 = 0.8631899952888489 + t4;
  const double t6 = vY * t5;
  const double t7 = 6.786799907684326 + t6;
  vUI = t7;
  const double t17 = vT * 7.28200006960833e-07;
  const double t18 = -0.014650000259280205 + t17;
  const double t19 = vT * t18;
  const double t20 = 86.01000213623047 + t19;
  const double t21 = (vT > 10400.0) ? 1.0 : 0.0;
  const double t22 = (t21 != 0.0) ? t20 : vUI;
  vUI = t22;
  const double t29 = 3.9999998989515007e-05 * vT;
  const double t30 = 5.46999979019165 + t29;
  vUII = t30;
  const double t32 = vT * 6.188000156726048e-08;
  const double t33 = -0.002219999907538295 + t32;
  const double t34 = vT * t33;
  const double t35 = 26.440000534057617 + t34;
  const double t36 = (vT > 18000.0) ? 1.0 : 0.0;
  const double t37 = (t36 != 0.0) ? t35 : vUII;
  vUII = t37;
  const double t44 = 1.1000000085914508e-05 * vT;
  const double t45 = 0.9110000133514404 + t44;
  const double t46 = (1.0 > t45) ? 1.0 : t45;
  vUIII = t46;
  const double t50 = vT * 2.616999950078025e-08;
  const double t51 = -0.001408000010997057 + t50;
  const double t52 = vT * t51;
  const double t53 = 19.139999389648438 + t52;
  const double t54 = (vT > 33300.0) ? 1.0 : 0.0;
  const double t55 = (t54 != 0.0) ? t53 : vUIII;
  vUIII = t55;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_14(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.0010380999883636832;
  const double t1 = 0.05730599910020828 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.2247599959373474 + t2;
  const double t4 = vY * t3;
  const double t5 = 4.225100040435791 + t4;
  vUI = t5;
  const double t6 = 3.0 * vY;
  const double t7 = t6 * 0.0010380999883636832;
  const double t8 = 0.11461199820041656 - t7;
  const double t9 = vY * t8;
  const double t10 = -0.2247599959373474 + t9;
  const double t11 = 0.0010000000474974513 * t10;
  const double t12 = PF_DIV(t11, vUI);
  vDUI = t12;
  const double t13 = 0.0005200000014156103 * vT;
  const double t14 = 1.559999942779541 + t13;
  const double t15 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t16 = (t15 != 0.0) ? t14 : vUI;
  vUI = t16;
  const double t17 = PF_DIV(0.0005200000014156103, vUI);
  const double t18 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t19 = (t18 != 0.0) ? t17 : vDUI;
  vDUI = t19;
  const double t20 = vY * 0.0035155999939888716;
  const double t21 = 0.07191299647092819 - t20;
  const double t22 = vY * t21;
  const double t23 = -0.5537099838256836 + t22;
  const double t24 = vY * t23;
  const double t25 = 2.2493999004364014 + t24;
  const double t26 = vY * t25;
  const double t27 = 4.41510009765625 + t26;
  vUII = t27;
  const double t28 = 4.0 * vY;
  const double t29 = t28 * 0.0035155999939888716;
  const double t30 = 0.21573898196220398 - t29;
  const double t31 = vY * t30;
  const double t32 = -1.1074199676513672 + t31;
  const double t33 = vY * t32;
  const double t34 = 2.2493999004364014 + t33;
  const double t35 = 0.0010000000474974513 * t34;
  const double t36 = PF_DIV(t35, vUII);
  vDUII = t36;
  const double t37 = 0.0005380000220611691 * vT;
  const double t38 = 4.619999885559082 + t37;
  const double t39 = (vT > 7250.0) ? 1.0 : 0.0;
  const double t40 = (t39 != 0.0) ? t38 : vUII;
  vUII = t40;
  const double t41 = PF_DIV(0.0005380000220611691, vUII);
  const double t42 = (vT > 7250.0) ? 1.0 : 0.0;
  const double t43 = (t42 != 0.0) ? t41 : vDUII;
  vDUII = t43;
  const double t44 = 3.400000059627928e-05 * vT;
  const double t45 = 5.59499979019165 + t44;
  vUIII = t45;
  const double t46 = PF_DIV(3.400000059627928e-05, vUIII);
  vDUIII = t46;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_14(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.0010380999883636832;
  const double t1 = 0.05730599910020828 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.2247599959373474 + t2;
  const double t4 = vY * t3;
  const double t5 = 4.225100040435791 + t4;
  vUI = t5;
  const double t13 = 0.0005200000014156103 * vT;
  const double t14 = 1.559999942779541 + t13;
  const double t15 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t16 = (t15 != 0.0) ? t14 : vUI;
  vUI = t16;
  const double t20 = vY * 0.0035155999939888716;
  const double t21 = 0.07191299647092819 - t20;
  const double t22 = vY * t21;
  const double t23 = -0.5537099838256836 + t22;
  const double t24 = vY * t23;
  const double t25 = 2.2493999004364014 + t24;
  const double t26 = vY * t25;
  const double t27 = 4.41510009765625 + t26;
  vUII = t27;
  const double t37 = 0.0005380000220611691 * vT;
  const double t38 = 4.619999885559082 + t37;
  const double t39 = (vT > 7250.0) ? 1.0 : 0.0;
  const double t40 = (t39 != 0.0) ? t38 : vUII;
  vUII = t40;
  const double t44 = 3.400000059627928e-05 * vT;
  const double t45 = 5.59499979019165 + t44;
  vUIII = t45;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_15(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.00021499999274965376 * vT;
  const double t1 = 7.5 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.00021499999274965376, vUI);
  vDUI = t2;
  const double t3 = vT * 2.124999980424036e-07;
  const double t4 = -0.004906000103801489 + t3;
  const double t5 = vT * t4;
  const double t6 = 38.7599983215332 + t5;
  const double t7 = (vT > 11600.0) ? 1.0 : 0.0;
  const double t8 = (t7 != 0.0) ? t6 : vUI;
  vUI = t8;
  const double t9 = 2.0 * vT;
  const double t10 = t9 * 2.124999980424036e-07;
  const double t11 = -0.004906000103801489 + t10;
  const double t12 = PF_DIV(t11, vUI);
  const double t13 = (vT > 11600.0) ? 1.0 : 0.0;
  const double t14 = (t13 != 0.0) ? t12 : vDUI;
  vDUI = t14;
  const double t15 = 0.00024300000222865492 * vT;
  const double t16 = 2.8450000286102295 + t15;
  vUII = t16;
  const double t17 = PF_DIV(0.00024300000222865492, vUII);
  vDUII = t17;
  const double t18 = vT * 1.3230000206476689e-08;
  const double t19 = -0.00016799999866634607 + t18;
  const double t20 = vT * t19;
  const double t21 = 6.406000137329102 + t20;
  const double t22 = (vT > 10500.0) ? 1.0 : 0.0;
  const double t23 = (t22 != 0.0) ? t21 : vUII;
  vUII = t23;
  const double t24 = vT * 2.0;
  const double t25 = t24 * 1.3230000206476689e-08;
  const double t26 = -0.00016799999866634607 + t25;
  const double t27 = PF_DIV(t26, vUII);
  const double t28 = (vT > 10500.0) ? 1.0 : 0.0;
  const double t29 = (t28 != 0.0) ? t27 : vDUII;
  vDUII = t29;
  const double t30 = 0.0001880000054370612 * vT;
  const double t31 = 7.380000114440918 + t30;
  vUIII = t31;
  const double t32 = PF_DIV(0.0001880000054370612, vUIII);
  vDUIII = t32;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_15(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.00021499999274965376 * vT;
  const double t1 = 7.5 + t0;
  vUI = t1;
  const double t3 = vT * 2.124999980424036e-07;
  const double t4 = -0.004906000103801489 + t3;
  const double t5 = vT * t4;
  const double t6 = 38.7599983215332 + t5;
  const double t7 = (vT > 11600.0) ? 1.0 : 0.0;
  const double t8 = (t7 != 0.0) ? t6 : vUI;
  vUI = t8;
  const double t15 = 0.00024300000222865492 * vT;
  const double t16 = 2.8450000286102295 + t15;
  vUII = t16;
  const double t18 = vT * 1.3230000206476689e-08;
  const double t19 = -0.00016799999866634607 + t18;
  const double t20 = vT * t19;
  const double t21 = 6.406000137329102 + t20;
  const double t22 = (vT > 10500.0) ? 1.0 : 0.0;
  const double t23 = (t22 != 0.0) ? t21 : vUII;
  vUII = t23;
  const double t30 = 0.0001880000054370612 * vT;
  const double t31 = 7.380000114440918 + t30;
  vUIII = t31;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_16(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 5.999999848427251e-05 * vT;
  const double t1 = 5.199999809265137 + t0;
  vUI = t1;
  const double t2 = PF_DIV(5.999999848427251e-05, vUI);
  vDUI = t2;
  const double t3 = 0.004800000227987766 * vT;
  const double t4 = -81.5999984741211 + t3;
  const double t5 = (vT > 18400.0) ? 1.0 : 0.0;
  const double t6 = (t5 != 0.0) ? t4 : vUI;
  vUI = t6;
  const double t7 = PF_DIV(0.004800000227987766, vUI);
  const double t8 = (vT > 18400.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vDUI;
  vDUI = t9;
  const double t10 = 0.00024300000222865492 * vT;
  const double t11 = 7.0 + t10;
  vUII = t11;
  const double t12 = PF_DIV(0.00024300000222865492, vUII);
  vDUII = t12;
  const double t13 = 0.00026199998683296144 * vT;
  const double t14 = 2.200000047683716 + t13;
  vUIII = t14;
  const double t15 = PF_DIV(0.00026199998683296144, vUIII);
  vDUIII = t15;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_16(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 5.999999848427251e-05 * vT;
  const double t1 = 5.199999809265137 + t0;
  vUI = t1;
  const double t3 = 0.004800000227987766 * vT;
  const double t4 = -81.5999984741211 + t3;
  const double t5 = (vT > 18400.0) ? 1.0 : 0.0;
  const double t6 = (t5 != 0.0) ? t4 : vUI;
  vUI = t6;
  const double t10 = 0.00024300000222865492 * vT;
  const double t11 = 7.0 + t10;
  vUII = t11;
  const double t13 = 0.00026199998683296144 * vT;
  const double t14 = 2.200000047683716 + t13;
  vUIII = t14;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_17(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 1.0;
  const double t0 = 3.7999998312443495e-05 * vT;
  const double t1 = 5.199999809265137 + t0;
  vUII = t1;
  const double t2 = PF_DIV(3.7999998312443495e-05, vUII);
  vDUII = t2;
  const double t3 = 0.0001554000045871362 * vT;
  const double t4 = 7.473999977111816 + t3;
  vUIII = t4;
  const double t5 = PF_DIV(0.0001554000045871362, vUIII);
  vDUIII = t5;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_17(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 1.0;
  const double t0 = 3.7999998312443495e-05 * vT;
  const double t1 = 5.199999809265137 + t0;
  vUII = t1;
  const double t3 = 0.0001554000045871362 * vT;
  const double t4 = 7.473999977111816 + t3;
  vUIII = t4;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_18(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.004093800205737352;
  const double t1 = 0.01743200048804283 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.023168999701738358 - t2;
  const double t4 = vY * t3;
  const double t5 = 1.9909000396728516 + t4;
  vUI = t5;
  const double t6 = vY * 3.0;
  const double t7 = t6 * 0.004093800205737352;
  const double t8 = 0.03486400097608566 - t7;
  const double t9 = vY * t8;
  const double t10 = 0.023168999701738358 - t9;
  const double t11 = 0.0010000000474974513 * t10;
  const double t12 = PF_DIV(t11, vUI);
  vDUI = t12;
  const double t13 = 0.002124000107869506 * vT;
  const double t14 = -9.930000305175781 + t13;
  const double t15 = (vT > 5800.0) ? 1.0 : 0.0;
  const double t16 = (t15 != 0.0) ? t14 : vUI;
  vUI = t16;
  const double t17 = PF_DIV(0.002124000107869506, vUI);
  const double t18 = (vT > 5800.0) ? 1.0 : 0.0;
  const double t19 = (t18 != 0.0) ? t17 : vDUI;
  vDUI = t19;
  vUII = 1.0;
  const double t20 = 1.9299999621580355e-05 * vT;
  const double t21 = 5.303999900817871 + t20;
  vUIII = t21;
  const double t22 = PF_DIV(1.9299999621580355e-05, vUIII);
  vDUIII = t22;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_18(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.004093800205737352;
  const double t1 = 0.01743200048804283 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.023168999701738358 - t2;
  const double t4 = vY * t3;
  const double t5 = 1.9909000396728516 + t4;
  vUI = t5;
  const double t13 = 0.002124000107869506 * vT;
  const double t14 = -9.930000305175781 + t13;
  const double t15 = (vT > 5800.0) ? 1.0 : 0.0;
  const double t16 = (t15 != 0.0) ? t14 : vUI;
  vUI = t16;
  vUII = 1.0;
  const double t20 = 1.9299999621580355e-05 * vT;
  const double t21 = 5.303999900817871 + t20;
  vUIII = t21;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_19(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.5085530281066895 * vX;
  const double t1 = 1.326861023902893 + t0;
  const double t2 = vX * t1;
  const double t3 = 1.6454559564590454 + t2;
  const double t4 = vX * t3;
  const double t5 = 5.004556179046631 + t4;
  const double t6 = vX * t5;
  const double t7 = -1.7312730550765991 - t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 1.0 + t8;
  vUI = t9;
  const double t10 = 2.034212112426758 * vX;
  const double t11 = 3.9805831909179688 + t10;
  const double t12 = vX * t11;
  const double t13 = 3.290911912918091 + t12;
  const double t14 = vX * t13;
  const double t15 = 5.004556179046631 + t14;
  const double t16 = vDX * t15;
  const double t17 = -t16;
  vDUI = t17;
  const double t18 = vUI - 1.0;
  const double t19 = vDUI * t18;
  const double t20 = PF_DIV(t19, vUI);
  vDUI = t20;
  const double t21 = 0.5396720170974731 * vX;
  const double t22 = 1.8907370567321777 + t21;
  const double t23 = vX * t22;
  const double t24 = 3.996088981628418 + t23;
  const double t25 = vX * t24;
  const double t26 = -1.5821119546890259 - t25;
  const double t27 = PF_EXP(t26);
  const double t28 = 2.0 + t27;
  vUII = t28;
  const double t29 = vX * 3.0;
  const double t30 = t29 * 0.5396720170974731;
  const double t31 = 3.7814741134643555 + t30;
  const double t32 = vX * t31;
  const double t33 = 3.996088981628418 + t32;
  const double t34 = vDX * t33;
  const double t35 = -t34;
  vDUII = t35;
  const double t36 = vUII - 2.0;
  const double t37 = vDUII * t36;
  const double t38 = PF_DIV(t37, vUII);
  vDUII = t38;
  vUIII = 1.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_19(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.5085530281066895 * vX;
  const double t1 = 1.326861023902893 + t0;
  const double t2 = vX * t1;
  const double t3 = 1.6454559564590454 + t2;
  const double t4 = vX * t3;
  const double t5 = 5.004556179046631 + t4;
  const double t6 = vX * t5;
  const double t7 = -1.7312730550765991 - t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 1.0 + t8;
  vUI = t9;
  const double t21 = 0.5396720170974731 * vX;
  const double t22 = 1.8907370567321777 + t21;
  const double t23 = vX * t22;
  const double t24 = 3.996088981628418 + t23;
  const double t25 = vX * t24;
  const double t26 = -1.5821119546890259 - t25;
  const double t27 = PF_EXP(t26);
  const double t28 = 2.0 + t27;
  vUII = t28;
  vUIII = 1.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_20(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.517795979976654 * vX;
  const double t1 = 1.1735039949417114 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.2391999959945679 + t2;
  const double t4 = vX * t3;
  const double t5 = 2.0715630054473877 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 4.0 + t6;
  vUI = t7;
  const double t8 = 3.0 * vX;
  const double t9 = t8 * 0.517795979976654;
  const double t10 = 2.347007989883423 + t9;
  const double t11 = vX * t10;
  const double t12 = -1.2391999959945679 + t11;
  const double t13 = vDX * t12;
  vDUI = t13;
  const double t14 = vUI - 4.0;
  const double t15 = vDUI * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = 0.05465799942612648 * vX;
  const double t18 = -0.5962380170822144 + t17;
  const double t19 = vX * t18;
  const double t20 = 2.9883620738983154 + t19;
  const double t21 = PF_EXP(t20);
  const double t22 = 3.0 + t21;
  vUII = t22;
  const double t23 = 2.0 * vX;
  const double t24 = t23 * 0.05465799942612648;
  const double t25 = -0.5962380170822144 + t24;
  const double t26 = vDX * t25;
  vDUII = t26;
  const double t27 = vUII - 3.0;
  const double t28 = vDUII * t27;
  const double t29 = PF_DIV(t28, vUII);
  vDUII = t29;
  vUIII = 10.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_20(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.517795979976654 * vX;
  const double t1 = 1.1735039949417114 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.2391999959945679 + t2;
  const double t4 = vX * t3;
  const double t5 = 2.0715630054473877 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 4.0 + t6;
  vUI = t7;
  const double t17 = 0.05465799942612648 * vX;
  const double t18 = -0.5962380170822144 + t17;
  const double t19 = vX * t18;
  const double t20 = 2.9883620738983154 + t19;
  const double t21 = PF_EXP(t20);
  const double t22 = 3.0 + t21;
  vUII = t22;
  vUIII = 10.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_21(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.27896299958229065 * vX;
  const double t1 = 0.7996129989624023 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.2277979850769043 + t2;
  const double t4 = vX * t3;
  const double t5 = 3.200453042984009 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 5.0 + t6;
  vUI = t7;
  const double t8 = 3.0 * vX;
  const double t9 = t8 * 0.27896299958229065;
  const double t10 = 1.5992259979248047 + t9;
  const double t11 = vX * t10;
  const double t12 = -1.2277979850769043 + t11;
  const double t13 = vDX * t12;
  vDUI = t13;
  const double t14 = vUI - 5.0;
  const double t15 = vDUI * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = vT * 5.818999966322735e-07;
  const double t18 = -0.0002838000073097646 + t17;
  const double t19 = vT * t18;
  const double t20 = 16.3700008392334 + t19;
  const double t21 = (vT < 5500.0) ? 1.0 : 0.0;
  const double t22 = (t21 != 0.0) ? t20 : vUI;
  vUI = t22;
  const double t23 = 2.0 * vT;
  const double t24 = t23 * 5.818999966322735e-07;
  const double t25 = -0.0002838000073097646 + t24;
  const double t26 = PF_DIV(t25, vUI);
  const double t27 = (vT < 5500.0) ? 1.0 : 0.0;
  const double t28 = (t27 != 0.0) ? t26 : vDUI;
  vDUI = t28;
  const double t29 = 0.11569300293922424 * vX;
  const double t30 = -0.5514310002326965 + t29;
  const double t31 = vX * t30;
  const double t32 = 3.9452900886535645 + t31;
  const double t33 = PF_EXP(t32);
  const double t34 = 4.0 + t33;
  vUII = t34;
  const double t35 = 2.0 * vX;
  const double t36 = t35 * 0.11569300293922424;
  const double t37 = -0.5514310002326965 + t36;
  const double t38 = vDX * t37;
  vDUII = t38;
  const double t39 = vUII - 4.0;
  const double t40 = vDUII * t39;
  const double t41 = PF_DIV(t40, vUII);
  vDUII = t41;
  const double t42 = 0.0008500000112690032 * vT;
  const double t43 = 16.399999618530273 + t42;
  vUIII = t43;
  const double t44 = PF_DIV(0.0008500000112690032, vUIII);
  vDUIII = t44;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_21(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.27896299958229065 * vX;
  const double t1 = 0.7996129989624023 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.2277979850769043 + t2;
  const double t4 = vX * t3;
  const double t5 = 3.200453042984009 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 5.0 + t6;
  vUI = t7;
  const double t17 = vT * 5.818999966322735e-07;
  const double t18 = -0.0002838000073097646 + t17;
  const double t19 = vT * t18;
  const double t20 = 16.3700008392334 + t19;
  const double t21 = (vT < 5500.0) ? 1.0 : 0.0;
  const double t22 = (t21 != 0.0) ? t20 : vUI;
  vUI = t22;
  const double t29 = 0.11569300293922424 * vX;
  const double t30 = -0.5514310002326965 + t29;
  const double t31 = vX * t30;
  const double t32 = 3.9452900886535645 + t31;
  const double t33 = PF_EXP(t32);
  const double t34 = 4.0 + t33;
  vUII = t34;
  const double t42 = 0.0008500000112690032 * vT;
  const double t43 = 16.399999618530273 + t42;
  vUIII = t43;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_22(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.16220000386238098 * vX;
  const double t1 = 0.724694013595581 + t0;
  const double t2 = vX * t1;
  const double t3 = -0.9063519835472107 + t2;
  const double t4 = vX * t3;
  const double t5 = 3.76961088180542 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 4.0 + t6;
  vUI = t7;
  const double t8 = 3.0 * vX;
  const double t9 = t8 * 0.16220000386238098;
  const double t10 = 1.449388027191162 + t9;
  const double t11 = vX * t10;
  const double t12 = -0.9063519835472107 + t11;
  const double t13 = vDX * t12;
  vDUI = t13;
  const double t14 = vUI - 4.0;
  const double t15 = vDUI * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = 0.21042999625205994 * vX;
  const double t18 = -0.7573710083961487 + t17;
  const double t19 = vX * t18;
  const double t20 = 3.7559170722961426 + t19;
  const double t21 = PF_EXP(t20);
  const double t22 = 1.0 + t21;
  vUII = t22;
  const double t23 = vX * 2.0;
  const double t24 = t23 * 0.21042999625205994;
  const double t25 = -0.7573710083961487 + t24;
  const double t26 = vDX * t25;
  vDUII = t26;
  const double t27 = vUII - 1.0;
  const double t28 = vDUII * t27;
  const double t29 = PF_DIV(t28, vUII);
  vDUII = t29;
  const double t30 = 0.010300000198185444 * vT;
  const double t31 = -18.0 + t30;
  vUIII = t31;
  const double t32 = PF_DIV(0.010300000198185444, vUIII);
  vDUIII = t32;
  const double t33 = 0.002400000113993883 * vT;
  const double t34 = (vT < 2250.0) ? 1.0 : 0.0;
  const double t35 = (t34 != 0.0) ? t33 : vUIII;
  vUIII = t35;
  const double t36 = PF_DIV(0.002400000113993883, vUIII);
  const double t37 = (vT < 2250.0) ? 1.0 : 0.0;
  const double t38 = (t37 != 0.0) ? t36 : vDUIII;
  vDUIII = t38;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_22(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.16220000386238098 * vX;
  const double t1 = 0.724694013595581 + t0;
  const double t2 = vX * t1;
  const double t3 = -0.9063519835472107 + t2;
  const double t4 = vX * t3;
  const double t5 = 3.76961088180542 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 4.0 + t6;
  vUI = t7;
  const double t17 = 0.21042999625205994 * vX;
  const double t18 = -0.7573710083961487 + t17;
  const double t19 = vX * t18;
  const double t20 = 3.7559170722961426 + t19;
  const double t21 = PF_EXP(t20);
  const double t22 = 1.0 + t21;
  vUII = t22;
  const double t30 = 0.010300000198185444 * vT;
  const double t31 = -18.0 + t30;
  vUIII = t31;
  const double t33 = 0.002400000113993883 * vT;
  const double t34 = (vT < 2250.0) ? 1.0 : 0.0;
  const double t35 = (t34 != 0.0) ? t33 : vUIII;
  vUIII = t35;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_23(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.09527000039815903 * vX;
  const double t1 = 0.15470899641513824 + t0;
  const double t2 = vX * t1;
  const double t3 = -2.923459053039551 + t2;
  const double t4 = vX * t3;
  const double t5 = 1.2250419855117798 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 7.0 + t6;
  vUI = t7;
  const double t8 = vX * 3.0;
  const double t9 = t8 * 0.09527000039815903;
  const double t10 = 0.3094179928302765 + t9;
  const double t11 = vX * t10;
  const double t12 = -2.923459053039551 + t11;
  const double t13 = vDX * t12;
  vDUI = t13;
  const double t14 = vUI - 7.0;
  const double t15 = vDUI * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = 0.2300730049610138 * vX;
  const double t18 = 1.0965479612350464 + t17;
  const double t19 = vX * t18;
  const double t20 = 4.143972873687744 + t19;
  const double t21 = vX * t20;
  const double t22 = 0.1287519931793213 - t21;
  const double t23 = PF_EXP(t22);
  const double t24 = 6.0 + t23;
  vUII = t24;
  const double t25 = 3.0 * vX;
  const double t26 = t25 * 0.2300730049610138;
  const double t27 = 2.1930959224700928 + t26;
  const double t28 = vX * t27;
  const double t29 = 4.143972873687744 + t28;
  const double t30 = vDX * t29;
  const double t31 = -t30;
  vDUII = t31;
  const double t32 = vUII - 6.0;
  const double t33 = vDUII * t32;
  const double t34 = PF_DIV(t33, vUII);
  vDUII = t34;
  const double t35 = 0.002099999925121665 * vT;
  const double t36 = 10.399999618530273 + t35;
  vUIII = t36;
  const double t37 = PF_DIV(0.002099999925121665, vUIII);
  vDUIII = t37;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_23(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.09527000039815903 * vX;
  const double t1 = 0.15470899641513824 + t0;
  const double t2 = vX * t1;
  const double t3 = -2.923459053039551 + t2;
  const double t4 = vX * t3;
  const double t5 = 1.2250419855117798 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 7.0 + t6;
  vUI = t7;
  const double t17 = 0.2300730049610138 * vX;
  const double t18 = 1.0965479612350464 + t17;
  const double t19 = vX * t18;
  const double t20 = 4.143972873687744 + t19;
  const double t21 = vX * t20;
  const double t22 = 0.1287519931793213 - t21;
  const double t23 = PF_EXP(t22);
  const double t24 = 6.0 + t23;
  vUII = t24;
  const double t35 = 0.002099999925121665 * vT;
  const double t36 = 10.399999618530273 + t35;
  vUIII = t36;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_24(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.2655569911003113 * vX;
  const double t1 = 1.0610549449920654 + t0;
  const double t2 = vX * t1;
  const double t3 = 2.136320114135742 + t2;
  const double t4 = vX * t3;
  const double t5 = 5.531251907348633 + t4;
  const double t6 = vX * t5;
  const double t7 = -0.869629979133606 - t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 6.0 + t8;
  vUI = t9;
  const double t10 = 1.0622279644012451 * vX;
  const double t11 = 3.1831648349761963 + t10;
  const double t12 = vX * t11;
  const double t13 = 4.272640228271484 + t12;
  const double t14 = vX * t13;
  const double t15 = 5.531251907348633 + t14;
  const double t16 = vDX * t15;
  const double t17 = -t16;
  vDUI = t17;
  const double t18 = vUI - 6.0;
  const double t19 = vDUI * t18;
  const double t20 = PF_DIV(t19, vUI);
  vDUI = t20;
  const double t21 = 0.1598220020532608 * vX;
  const double t22 = 0.814674973487854 + t21;
  const double t23 = vX * t22;
  const double t24 = 3.77278995513916 + t23;
  const double t25 = vX * t24;
  const double t26 = -0.28296101093292236 - t25;
  const double t27 = PF_EXP(t26);
  const double t28 = 7.0 + t27;
  vUII = t28;
  const double t29 = 3.0 * vX;
  const double t30 = t29 * 0.1598220020532608;
  const double t31 = 1.629349946975708 + t30;
  const double t32 = vX * t31;
  const double t33 = 3.77278995513916 + t32;
  const double t34 = vDX * t33;
  const double t35 = -t34;
  vDUII = t35;
  const double t36 = vUII - 7.0;
  const double t37 = vDUII * t36;
  const double t38 = PF_DIV(t37, vUII);
  vDUII = t38;
  vUIII = 10.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_24(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.2655569911003113 * vX;
  const double t1 = 1.0610549449920654 + t0;
  const double t2 = vX * t1;
  const double t3 = 2.136320114135742 + t2;
  const double t4 = vX * t3;
  const double t5 = 5.531251907348633 + t4;
  const double t6 = vX * t5;
  const double t7 = -0.869629979133606 - t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 6.0 + t8;
  vUI = t9;
  const double t21 = 0.1598220020532608 * vX;
  const double t22 = 0.814674973487854 + t21;
  const double t23 = vX * t22;
  const double t24 = 3.77278995513916 + t23;
  const double t25 = vX * t24;
  const double t26 = -0.28296101093292236 - t25;
  const double t27 = PF_EXP(t26);
  const double t28 = 7.0 + t27;
  vUII = t28;
  vUIII = 10.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_25(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.11821799725294113 * vX;
  const double t1 = 0.7602699995040894 + t0;
  const double t2 = vX * t1;
  const double t3 = -0.9797449707984924 + t2;
  const double t4 = vX * t3;
  const double t5 = 2.930047035217285 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 9.0 + t6;
  vUI = t7;
  const double t8 = 3.0 * vX;
  const double t9 = t8 * 0.11821799725294113;
  const double t10 = 1.5205399990081787 + t9;
  const double t11 = vX * t10;
  const double t12 = -0.9797449707984924 + t11;
  const double t13 = vDX * t12;
  vDUI = t13;
  const double t14 = vUI - 9.0;
  const double t15 = vDUI * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = vT * 2.0400000266818097e-07;
  const double t18 = 0.001306000049225986 + t17;
  const double t19 = vT * t18;
  const double t20 = 15.850000381469727 + t19;
  const double t21 = (vT < 4000.0) ? 1.0 : 0.0;
  const double t22 = (t21 != 0.0) ? t20 : vUI;
  vUI = t22;
  const double t23 = 2.0 * vT;
  const double t24 = t23 * 2.0400000266818097e-07;
  const double t25 = 0.001306000049225986 + t24;
  const double t26 = PF_DIV(t25, vUI);
  const double t27 = (vT < 4000.0) ? 1.0 : 0.0;
  const double t28 = (t27 != 0.0) ? t26 : vDUI;
  vDUI = t28;
  const double t29 = vT * 1.247699970008398e-06;
  const double t30 = -0.009592199698090553 + t29;
  const double t31 = vT * t30;
  const double t32 = 39.14899826049805 + t31;
  const double t33 = (vT > 9000.0) ? 1.0 : 0.0;
  const double t34 = (t33 != 0.0) ? t32 : vUI;
  vUI = t34;
  const double t35 = 2.0 * vT;
  const double t36 = t35 * 1.247699970008398e-06;
  const double t37 = -0.009592199698090553 + t36;
  const double t38 = PF_DIV(t37, vUI);
  const double t39 = (vT > 9000.0) ? 1.0 : 0.0;
  const double t40 = (t39 != 0.0) ? t38 : vDUI;
  vDUI = t40;
  const double t41 = 0.28098198771476746 * vX;
  const double t42 = -0.612093985080719 + t41;
  const double t43 = vX * t42;
  const double t44 = 3.5015969276428223 + t43;
  const double t45 = PF_EXP(t44);
  const double t46 = 10.0 + t45;
  vUII = t46;
  const double t47 = 2.0 * vX;
  const double t48 = t47 * 0.28098198771476746;
  const double t49 = -0.612093985080719 + t48;
  const double t50 = vDX * t49;
  vDUII = t50;
  const double t51 = vUII - 10.0;
  const double t52 = vDUII * t51;
  const double t53 = PF_DIV(t52, vUII);
  vDUII = t53;
  const double t54 = vT * 5.156700240149803e-07;
  const double t55 = -0.006110399961471558 + t54;
  const double t56 = vT * t55;
  const double t57 = 68.35600280761719 + t56;
  const double t58 = (vT > 18000.0) ? 1.0 : 0.0;
  const double t59 = (t58 != 0.0) ? t57 : vUII;
  vUII = t59;
  const double t60 = 2.0 * vT;
  const double t61 = t60 * 5.156700240149803e-07;
  const double t62 = -0.006110399961471558 + t61;
  const double t63 = PF_DIV(t62, vUII);
  const double t64 = (vT > 18000.0) ? 1.0 : 0.0;
  const double t65 = (t64 != 0.0) ? t63 : vDUII;
  vDUII = t65;
  const double t66 = vT * 5.751400067310897e-08;
  const double t67 = 0.0005504799773916602 + t66;
  const double t68 = vT * t67;
  const double t69 = 17.336000442504883 + t68;
  vUIII = t69;
  const double t70 = 2.0 * vT;
  const double t71 = t70 * 5.751400067310897e-08;
  const double t72 = 0.0005504799773916602 + t71;
  const double t73 = PF_DIV(t72, vUIII);
  vDUIII = t73;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_25(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.11821799725294113 * vX;
  const double t1 = 0.7602699995040894 + t0;
  const double t2 = vX * t1;
  const double t3 = -0.9797449707984924 + t2;
  const double t4 = vX * t3;
  const double t5 = 2.930047035217285 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 9.0 + t6;
  vUI = t7;
  const double t17 = vT * 2.0400000266818097e-07;
  const double t18 = 0.001306000049225986 + t17;
  const double t19 = vT * t18;
  const double t20 = 15.850000381469727 + t19;
  const double t21 = (vT < 4000.0) ? 1.0 : 0.0;
  const double t22 = (t21 != 0.0) ? t20 : vUI;
  vUI = t22;
  const double t29 = vT * 1.247699970008398e-06;
  const double t30 = -0.009592199698090553 + t29;
  const double t31 = vT * t30;
  const double t32 = 39.14899826049805 + t31;
  const double t33 = (vT > 9000.0) ? 1.0 : 0.0;
  const double t34 = (t33 != 0.0) ? t32 : vUI;
  vUI = t34;
  const double t41 = 0.28098198771476746 * vX;
  const double t42 = -0.612093985080719 + t41;
  const double t43 = vX * t42;
  const double t44 = 3.5015969276428223 + t43;
  const double t45 = PF_EXP(t44);
  const double t46 = 10.0 + t45;
  vUII = t46;
  const double t54 = vT * 5.156700240149803e-07;
  const double t55 = -0.006110399961471558 + t54;
  const double t56 = vT * t55;
  const double t57 = 68.35600280761719 + t56;
  const double t58 = (vT > 18000.0) ? 1.0 : 0.0;
  const double t59 = (t58 != 0.0) ? t57 : vUII;
  vUII = t59;
  const double t66 = vT * 5.751400067310897e-08;
  const double t67 = 0.0005504799773916602 + t66;
  const double t68 = vT * t67;
  const double t69 = 17.336000442504883 + t68;
  vUIII = t69;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_26(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.004900000058114529 * vT;
  const double t1 = 8.649999618530273 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.004900000058114529, vUI);
  vDUI = t2;
  const double t3 = 0.0035800000187009573 * vT;
  const double t4 = 11.199999809265137 + t3;
  vUII = t4;
  const double t5 = PF_DIV(0.0035800000187009573, vUII);
  vDUII = t5;
  const double t6 = 0.0014199999859556556 * vT;
  const double t7 = 15.0 + t6;
  vUIII = t7;
  const double t8 = PF_DIV(0.0014199999859556556, vUIII);
  vDUIII = t8;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_26(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.004900000058114529 * vT;
  const double t1 = 8.649999618530273 + t0;
  vUI = t1;
  const double t3 = 0.0035800000187009573 * vT;
  const double t4 = 11.199999809265137 + t3;
  vUII = t4;
  const double t6 = 0.0014199999859556556 * vT;
  const double t7 = 15.0 + t6;
  vUIII = t7;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_27(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.2784680128097534 * vX;
  const double t1 = 0.07749799638986588 - t0;
  const double t2 = vX * t1;
  const double t3 = -0.40132299065589905 + t2;
  const double t4 = vX * t3;
  const double t5 = 3.084552049636841 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 9.0 + t6;
  vUI = t7;
  const double t8 = 3.0 * vX;
  const double t9 = t8 * 0.2784680128097534;
  const double t10 = 0.15499599277973175 - t9;
  const double t11 = vX * t10;
  const double t12 = -0.40132299065589905 + t11;
  const double t13 = vDX * t12;
  vDUI = t13;
  const double t14 = vUI - 9.0;
  const double t15 = vDUI * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = 0.11565399914979935 * vX;
  const double t18 = 1.528965950012207 + t17;
  const double t19 = vX * t18;
  const double t20 = 1.593047022819519 - t19;
  const double t21 = PF_EXP(t20);
  const double t22 = 6.0 + t21;
  vUII = t22;
  const double t23 = 2.0 * vX;
  const double t24 = t23 * 0.11565399914979935;
  const double t25 = 1.528965950012207 + t24;
  const double t26 = vDX * t25;
  const double t27 = -t26;
  vDUII = t27;
  const double t28 = vUII - 6.0;
  const double t29 = vDUII * t28;
  const double t30 = PF_DIV(t29, vUII);
  vDUII = t30;
  const double t31 = 0.0006900000153109431 * vT;
  const double t32 = 13.300000190734863 + t31;
  vUIII = t32;
  const double t33 = PF_DIV(0.0006900000153109431, vUIII);
  vDUIII = t33;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_27(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.2784680128097534 * vX;
  const double t1 = 0.07749799638986588 - t0;
  const double t2 = vX * t1;
  const double t3 = -0.40132299065589905 + t2;
  const double t4 = vX * t3;
  const double t5 = 3.084552049636841 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 9.0 + t6;
  vUI = t7;
  const double t17 = 0.11565399914979935 * vX;
  const double t18 = 1.528965950012207 + t17;
  const double t19 = vX * t18;
  const double t20 = 1.593047022819519 - t19;
  const double t21 = PF_EXP(t20);
  const double t22 = 6.0 + t21;
  vUII = t22;
  const double t31 = 0.0006900000153109431 * vT;
  const double t32 = 13.300000190734863 + t31;
  vUIII = t32;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_28(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.00015100000018719584 * vT;
  const double t1 = 1.5 + t0;
  const double t2 = (2.0 > t1) ? 2.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(0.00015100000018719584, vUI);
  const double t4 = (vUI != 2.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  const double t6 = 0.0004579999949783087 * vT;
  const double t7 = -0.30000001192092896 + t6;
  const double t8 = (vT > 6250.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t10 = PF_DIV(0.0004579999949783087, vUI);
  const double t11 = (vT > 6250.0) ? 1.0 : 0.0;
  const double t12 = (t11 != 0.0) ? t10 : vDUI;
  vDUI = t12;
  const double t13 = 0.00014899999951012433 * vT;
  const double t14 = 0.2199999988079071 + t13;
  const double t15 = (1.0 > t14) ? 1.0 : t14;
  vUII = t15;
  const double t16 = PF_DIV(0.00014899999951012433, vUII);
  const double t17 = (vUII != 1.0) ? 1.0 : 0.0;
  const double t18 = (t17 != 0.0) ? t16 : vDUII;
  vDUII = t18;
  const double t19 = 9.40000027185306e-05 * vT;
  const double t20 = 8.024999618530273 + t19;
  vUIII = t20;
  const double t21 = PF_DIV(9.40000027185306e-05, vUIII);
  vDUIII = t21;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_28(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.00015100000018719584 * vT;
  const double t1 = 1.5 + t0;
  const double t2 = (2.0 > t1) ? 2.0 : t1;
  vUI = t2;
  const double t6 = 0.0004579999949783087 * vT;
  const double t7 = -0.30000001192092896 + t6;
  const double t8 = (vT > 6250.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t13 = 0.00014899999951012433 * vT;
  const double t14 = 0.2199999988079071 + t13;
  const double t15 = (1.0 > t14) ? 1.0 : t14;
  vUII = t15;
  const double t19 = 9.40000027185306e-05 * vT;
  const double t20 = 8.024999618530273 + t19;
  vUIII = t20;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_29(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 5.109999983687885e-05 * vT;
  const double t1 = 0.6320000290870667 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(5.109999983687885e-05, vUI);
  const double t4 = (vUI != 1.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  vUII = 2.0;
  vUIII = 1.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_29(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 5.109999983687885e-05 * vT;
  const double t1 = 0.6320000290870667 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  vUII = 2.0;
  vUIII = 1.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_30(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.0025053999852389097;
  const double t1 = 0.05487599968910217 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.4643000066280365 + t2;
  const double t4 = vY * t3;
  const double t5 = 1.9337999820709229 + t4;
  const double t6 = vY * t5;
  const double t7 = 1.7930999994277954 + t6;
  vUI = t7;
  const double t8 = vY * 4.0;
  const double t9 = t8 * 0.0025053999852389097;
  const double t10 = 0.16462799906730652 - t9;
  const double t11 = vY * t10;
  const double t12 = -0.928600013256073 + t11;
  const double t13 = vY * t12;
  const double t14 = 1.9337999820709229 + t13;
  const double t15 = 0.0010000000474974513 * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = 0.00020300000323913991 * vT;
  const double t18 = 4.179999828338623 + t17;
  const double t19 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t20 = (t19 != 0.0) ? t18 : vUI;
  vUI = t20;
  const double t21 = PF_DIV(0.00020300000323913991, vUI);
  const double t22 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t23 = (t22 != 0.0) ? t21 : vDUI;
  vDUI = t23;
  vUII = 1.0;
  vUIII = 2.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_30(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.0025053999852389097;
  const double t1 = 0.05487599968910217 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.4643000066280365 + t2;
  const double t4 = vY * t3;
  const double t5 = 1.9337999820709229 + t4;
  const double t6 = vY * t5;
  const double t7 = 1.7930999994277954 + t6;
  vUI = t7;
  const double t17 = 0.00020300000323913991 * vT;
  const double t18 = 4.179999828338623 + t17;
  const double t19 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t20 = (t19 != 0.0) ? t18 : vUI;
  vUI = t20;
  vUII = 1.0;
  vUIII = 2.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_31(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0004079999926034361 * vT;
  const double t1 = 6.119999885559082 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.0004079999926034361, vUI);
  vDUI = t2;
  const double t3 = 0.00017800000205170363 * vT;
  const double t4 = 3.444999933242798 + t3;
  vUII = t4;
  const double t5 = PF_DIV(0.00017800000205170363, vUII);
  vDUII = t5;
  vUIII = 1.100000023841858;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_31(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0004079999926034361 * vT;
  const double t1 = 6.119999885559082 + t0;
  vUI = t1;
  const double t3 = 0.00017800000205170363 * vT;
  const double t4 = 3.444999933242798 + t3;
  vUII = t4;
  vUIII = 1.100000023841858;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_32(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0003650000144261867 * vT;
  const double t1 = 2.6500000953674316 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.0003650000144261867, vUI);
  vDUI = t2;
  const double t3 = vY * 0.0011608999921008945;
  const double t4 = 0.030408000573515892 - t3;
  const double t5 = vY * t4;
  const double t6 = -0.33382999897003174 + t5;
  const double t7 = vY * t6;
  const double t8 = 2.2839999198913574 + t7;
  const double t9 = vY * t8;
  const double t10 = -0.25383999943733215 + t9;
  vUII = t10;
  const double t11 = 4.0 * vY;
  const double t12 = t11 * 0.0011608999921008945;
  const double t13 = 0.09122399985790253 - t12;
  const double t14 = vY * t13;
  const double t15 = -0.6676599979400635 + t14;
  const double t16 = vY * t15;
  const double t17 = 2.2839999198913574 + t16;
  const double t18 = 0.0010000000474974513 * t17;
  const double t19 = PF_DIV(t18, vUII);
  vDUII = t19;
  const double t20 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t21 = (t20 != 0.0) ? 8.0 : vUII;
  vUII = t21;
  const double t22 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t23 = (t22 != 0.0) ? 0.0 : vDUII;
  vDUII = t23;
  vUIII = 8.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_32(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0003650000144261867 * vT;
  const double t1 = 2.6500000953674316 + t0;
  vUI = t1;
  const double t3 = vY * 0.0011608999921008945;
  const double t4 = 0.030408000573515892 - t3;
  const double t5 = vY * t4;
  const double t6 = -0.33382999897003174 + t5;
  const double t7 = vY * t6;
  const double t8 = 2.2839999198913574 + t7;
  const double t9 = vY * t8;
  const double t10 = -0.25383999943733215 + t9;
  vUII = t10;
  const double t20 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t21 = (t20 != 0.0) ? 8.0 : vUII;
  vUII = t21;
  vUIII = 8.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_33(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.00017100000695791095 * vT;
  const double t1 = 6.340000152587891 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.00017100000695791095, vUI);
  vDUI = t2;
  const double t3 = 0.03205300122499466 * vY;
  const double t4 = -0.1539199948310852 + t3;
  const double t5 = vY * t4;
  const double t6 = 4.178599834442139 + t5;
  vUII = t6;
  const double t7 = 0.03205300122499466 * vY;
  const double t8 = t7 * 2.0;
  const double t9 = -0.1539199948310852 + t8;
  const double t10 = 0.0010000000474974513 * t9;
  const double t11 = PF_DIV(t10, vUII);
  vDUII = t11;
  vUIII = 8.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_33(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.00017100000695791095 * vT;
  const double t1 = 6.340000152587891 + t0;
  vUI = t1;
  const double t3 = 0.03205300122499466 * vY;
  const double t4 = -0.1539199948310852 + t3;
  const double t5 = vY * t4;
  const double t6 = 4.178599834442139 + t5;
  vUII = t6;
  vUIII = 8.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_34(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.00011200000153621659 * vT;
  const double t1 = 4.119999885559082 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.00011200000153621659, vUI);
  vDUI = t2;
  const double t3 = 0.000307999987853691 * vT;
  const double t4 = 5.21999979019165 + t3;
  vUII = t4;
  const double t5 = PF_DIV(0.000307999987853691, vUII);
  vDUII = t5;
  const double t6 = 0.0002859999949578196 * vT;
  const double t7 = 2.299999952316284 + t6;
  vUIII = t7;
  const double t8 = PF_DIV(0.0002859999949578196, vUIII);
  vDUIII = t8;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_34(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.00011200000153621659 * vT;
  const double t1 = 4.119999885559082 + t0;
  vUI = t1;
  const double t3 = 0.000307999987853691 * vT;
  const double t4 = 5.21999979019165 + t3;
  vUII = t4;
  const double t6 = 0.0002859999949578196 * vT;
  const double t7 = 2.299999952316284 + t6;
  vUIII = t7;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_35(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 1.0;
  const double t0 = 7.400000322377309e-05 * vT;
  const double t1 = 4.110000133514404 + t0;
  vUII = t1;
  const double t2 = PF_DIV(7.400000322377309e-05, vUII);
  vDUII = t2;
  const double t3 = 0.0002229999954579398 * vT;
  const double t4 = 5.349999904632568 + t3;
  vUIII = t4;
  const double t5 = PF_DIV(0.0002229999954579398, vUIII);
  vDUIII = t5;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_35(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 1.0;
  const double t0 = 7.400000322377309e-05 * vT;
  const double t1 = 4.110000133514404 + t0;
  vUII = t1;
  const double t3 = 0.0002229999954579398 * vT;
  const double t4 = 5.349999904632568 + t3;
  vUIII = t4;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_36(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0001939999929163605 * vT;
  const double t1 = 1.3799999952316284 + t0;
  const double t2 = (2.0 > t1) ? 2.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(0.0001939999929163605, vUI);
  const double t4 = (vUI != 2.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  const double t6 = 0.00279000005684793 * vT;
  const double t7 = -14.899999618530273 + t6;
  const double t8 = (vT > 6250.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t10 = PF_DIV(0.00279000005684793, vUI);
  const double t11 = (vT > 6250.0) ? 1.0 : 0.0;
  const double t12 = (t11 != 0.0) ? t10 : vDUI;
  vDUI = t12;
  vUII = 1.0;
  const double t13 = 4.8499998229090124e-05 * vT;
  const double t14 = 4.206999778747559 + t13;
  vUIII = t14;
  const double t15 = PF_DIV(4.8499998229090124e-05, vUIII);
  vDUIII = t15;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_36(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0001939999929163605 * vT;
  const double t1 = 1.3799999952316284 + t0;
  const double t2 = (2.0 > t1) ? 2.0 : t1;
  vUI = t2;
  const double t6 = 0.00279000005684793 * vT;
  const double t7 = -14.899999618530273 + t6;
  const double t8 = (vT > 6250.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  vUII = 1.0;
  const double t13 = 4.8499998229090124e-05 * vT;
  const double t14 = 4.206999778747559 + t13;
  vUIII = t14;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_37(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.0010230999905616045;
  const double t1 = 0.021423999220132828 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.10745999962091446 + t2;
  const double t4 = vY * t3;
  const double t5 = 0.20148000121116638 + t4;
  const double t6 = vY * t5;
  const double t7 = 0.8712700009346008 + t6;
  vUI = t7;
  const double t8 = vY * 0.0010230999905616045;
  const double t9 = t8 * 4.0;
  const double t10 = 0.06427200138568878 - t9;
  const double t11 = vY * t10;
  const double t12 = -0.21491999924182892 + t11;
  const double t13 = vY * t12;
  const double t14 = 0.20148000121116638 + t13;
  const double t15 = 0.0010000000474974513 * t14;
  vDUI = t15;
  const double t16 = PF_DIV(vDUI, vUI);
  vDUI = t16;
  const double t17 = 0.0012240000069141388 * vT;
  const double t18 = -6.119999885559082 + t17;
  const double t19 = (vT > 6500.0) ? 1.0 : 0.0;
  const double t20 = (t19 != 0.0) ? t18 : vUI;
  vUI = t20;
  const double t21 = PF_DIV(0.0012240000069141388, vUI);
  const double t22 = (vT > 6500.0) ? 1.0 : 0.0;
  const double t23 = (t22 != 0.0) ? t21 : vDUI;
  vDUI = t23;
  const double t24 = 0.00026000000070780516 * vT;
  const double t25 = 0.8399999737739563 + t24;
  const double t26 = (2.0 > t25) ? 2.0 : t25;
  vUII = t26;
  const double t27 = PF_DIV(0.00026000000070780516, vUII);
  const double t28 = (vUII != 2.0) ? 1.0 : 0.0;
  const double t29 = (t28 != 0.0) ? t27 : vDUII;
  vDUII = t29;
  vUIII = 1.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_37(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.0010230999905616045;
  const double t1 = 0.021423999220132828 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.10745999962091446 + t2;
  const double t4 = vY * t3;
  const double t5 = 0.20148000121116638 + t4;
  const double t6 = vY * t5;
  const double t7 = 0.8712700009346008 + t6;
  vUI = t7;
  const double t17 = 0.0012240000069141388 * vT;
  const double t18 = -6.119999885559082 + t17;
  const double t19 = (vT > 6500.0) ? 1.0 : 0.0;
  const double t20 = (t19 != 0.0) ? t18 : vUI;
  vUI = t20;
  const double t24 = 0.00026000000070780516 * vT;
  const double t25 = 0.8399999737739563 + t24;
  const double t26 = (2.0 > t25) ? 2.0 : t25;
  vUII = t26;
  vUIII = 1.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_38(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.002580000087618828 * vT;
  const double t1 = 0.20000000298023224 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.002580000087618828, vUI);
  vDUI = t2;
  const double t3 = 0.0018550000386312604 * vT;
  const double t4 = 7.150000095367432 + t3;
  vUII = t4;
  const double t5 = PF_DIV(0.0018550000386312604, vUII);
  vDUII = t5;
  const double t6 = 9.899999713525176e-05 * vT;
  const double t7 = 9.710000038146973 + t6;
  vUIII = t7;
  const double t8 = PF_DIV(9.899999713525176e-05, vUIII);
  vDUIII = t8;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_38(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.002580000087618828 * vT;
  const double t1 = 0.20000000298023224 + t0;
  vUI = t1;
  const double t3 = 0.0018550000386312604 * vT;
  const double t4 = 7.150000095367432 + t3;
  vUII = t4;
  const double t6 = 9.899999713525176e-05 * vT;
  const double t7 = 9.710000038146973 + t6;
  vUIII = t7;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_39(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vT * 2.198999936808832e-06;
  const double t1 = -0.01865999959409237 + t0;
  const double t2 = vT * t1;
  const double t3 = 76.30999755859375 + t2;
  vUI = t3;
  const double t4 = vT * 2.198999936808832e-06;
  const double t5 = t4 * 2.0;
  const double t6 = -0.01865999959409237 + t5;
  const double t7 = PF_DIV(t6, vUI);
  vDUI = t7;
  const double t8 = vT * 5.385999770624039e-07;
  const double t9 = 0.0028059999458491802 + t8;
  const double t10 = vT * t9;
  const double t11 = 6.800000190734863 + t10;
  const double t12 = (vT < 6236.0) ? 1.0 : 0.0;
  const double t13 = (t12 != 0.0) ? t11 : vUI;
  vUI = t13;
  const double t14 = vT * 5.385999770624039e-07;
  const double t15 = t14 * 2.0;
  const double t16 = 0.0028059999458491802 + t15;
  const double t17 = PF_DIV(t16, vUI);
  const double t18 = (vT < 6236.0) ? 1.0 : 0.0;
  const double t19 = (t18 != 0.0) ? t17 : vDUI;
  vDUI = t19;
  const double t20 = 0.9065020084381104 * vX;
  const double t21 = 3.7213289737701416 - t20;
  const double t22 = PF_EXP(t21);
  const double t23 = 4.0 + t22;
  vUII = t23;
  const double t24 = vDX * 0.9065020084381104;
  const double t25 = -t24;
  vDUII = t25;
  const double t26 = vUII - 4.0;
  const double t27 = vDUII * t26;
  const double t28 = PF_DIV(t27, vUII);
  vDUII = t28;
  const double t29 = 0.0013849999522790313 * vT;
  const double t30 = 12.300000190734863 + t29;
  vUIII = t30;
  const double t31 = PF_DIV(0.0013849999522790313, vUIII);
  vDUIII = t31;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_39(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vT * 2.198999936808832e-06;
  const double t1 = -0.01865999959409237 + t0;
  const double t2 = vT * t1;
  const double t3 = 76.30999755859375 + t2;
  vUI = t3;
  const double t8 = vT * 5.385999770624039e-07;
  const double t9 = 0.0028059999458491802 + t8;
  const double t10 = vT * t9;
  const double t11 = 6.800000190734863 + t10;
  const double t12 = (vT < 6236.0) ? 1.0 : 0.0;
  const double t13 = (t12 != 0.0) ? t11 : vUI;
  vUI = t13;
  const double t20 = 0.9065020084381104 * vX;
  const double t21 = 3.7213289737701416 - t20;
  const double t22 = PF_EXP(t21);
  const double t23 = 4.0 + t22;
  vUII = t23;
  const double t29 = 0.0013849999522790313 * vT;
  const double t30 = 12.300000190734863 + t29;
  vUIII = t30;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_40(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.014299999922513962 * vT;
  const double t1 = -19.0 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(0.014299999922513962, vUI);
  const double t4 = (vUI != 1.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  const double t6 = 0.0101500004529953 * vT;
  const double t7 = -4.0 + t6;
  vUII = t7;
  const double t8 = PF_DIV(0.0101500004529953, vUII);
  vDUII = t8;
  vUIII = 25.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_40(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.014299999922513962 * vT;
  const double t1 = -19.0 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  const double t6 = 0.0101500004529953 * vT;
  const double t7 = -4.0 + t6;
  vUII = t7;
  vUIII = 25.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_41(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.001500000013038516 * vT;
  const double t1 = 2.0999999046325684 + t0;
  const double t2 = (7.0 > t1) ? 7.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(0.001500000013038516, vUI);
  const double t4 = (vUI != 7.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  const double t6 = 0.007280000019818544 * vT;
  const double t7 = -38.099998474121094 + t6;
  const double t8 = (vT > 7000.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t10 = PF_DIV(0.007280000019818544, vUI);
  const double t11 = (vT > 7000.0) ? 1.0 : 0.0;
  const double t12 = (t11 != 0.0) ? t10 : vDUI;
  vDUI = t12;
  const double t13 = 0.0011699999449774623 * vT;
  const double t14 = 1.25 + t13;
  vUII = t14;
  const double t15 = PF_DIV(0.0011699999449774623, vUII);
  vDUII = t15;
  const double t16 = 0.00547999981790781 * vT;
  const double t17 = -28.5 + t16;
  const double t18 = (vT > 6900.0) ? 1.0 : 0.0;
  const double t19 = (t18 != 0.0) ? t17 : vUII;
  vUII = t19;
  const double t20 = PF_DIV(0.00547999981790781, vUII);
  const double t21 = (vT > 6900.0) ? 1.0 : 0.0;
  const double t22 = (t21 != 0.0) ? t20 : vDUII;
  vDUII = t22;
  const double t23 = 0.0001463999942643568 * vT;
  const double t24 = 24.040000915527344 + t23;
  vUIII = t24;
  const double t25 = PF_DIV(0.0001463999942643568, vUIII);
  vDUIII = t25;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_41(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.001500000013038516 * vT;
  const double t1 = 2.0999999046325684 + t0;
  const double t2 = (7.0 > t1) ? 7.0 : t1;
  vUI = t2;
  const double t6 = 0.007280000019818544 * vT;
  const double t7 = -38.099998474121094 + t6;
  const double t8 = (vT > 7000.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t13 = 0.0011699999449774623 * vT;
  const double t14 = 1.25 + t13;
  vUII = t14;
  const double t16 = 0.00547999981790781 * vT;
  const double t17 = -28.5 + t16;
  const double t18 = (vT > 6900.0) ? 1.0 : 0.0;
  const double t19 = (t18 != 0.0) ? t17 : vUII;
  vUII = t19;
  const double t23 = 0.0001463999942643568 * vT;
  const double t24 = 24.040000915527344 + t23;
  vUIII = t24;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_42(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.0021538001019507647;
  const double t1 = 0.04840100184082985 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.40779998898506165 + t2;
  const double t4 = vY * t3;
  const double t5 = 1.652500033378601 + t4;
  const double t6 = vY * t5;
  const double t7 = 0.3064799904823303 + t6;
  const double t8 = vY * t7;
  const double t9 = 4.439000129699707 + t8;
  vUI = t9;
  const double t10 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t11 = (t10 != 0.0) ? 24.0 : vUI;
  vUI = t11;
  const double t12 = vY * 0.0021538001019507647;
  const double t13 = t12 * 5.0;
  const double t14 = 0.1936040073633194 - t13;
  const double t15 = vY * t14;
  const double t16 = -1.2233999967575073 + t15;
  const double t17 = vY * t16;
  const double t18 = 3.305000066757202 + t17;
  const double t19 = vY * t18;
  const double t20 = 0.3064799904823303 + t19;
  const double t21 = 0.0010000000474974513 * t20;
  const double t22 = PF_DIV(t21, vUI);
  const double t23 = (vT <= 6000.0) ? 1.0 : 0.0;
  const double t24 = (t23 != 0.0) ? t22 : vDUI;
  vDUI = t24;
  const double t25 = vY * 0.001908699981868267;
  const double t26 = 0.04965599998831749 - t25;
  const double t27 = vY * t26;
  const double t28 = -0.5019999742507935 + t27;
  const double t29 = vY * t28;
  const double t30 = 2.36899995803833 + t29;
  const double t31 = vY * t30;
  const double t32 = -2.9630000591278076 + t31;
  const double t33 = vY * t32;
  const double t34 = 8.109600067138672 + t33;
  vUII = t34;
  const double t35 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t36 = (t35 != 0.0) ? 17.0 : vUII;
  vUII = t36;
  const double t37 = vY * 0.001908699981868267;
  const double t38 = t37 * 5.0;
  const double t39 = 0.19862399995326996 - t38;
  const double t40 = vY * t39;
  const double t41 = -1.5059999227523804 + t40;
  const double t42 = vY * t41;
  const double t43 = 4.73799991607666 + t42;
  const double t44 = vY * t43;
  const double t45 = -2.9630000591278076 + t44;
  const double t46 = 0.0010000000474974513 * t45;
  const double t47 = PF_DIV(t46, vUII);
  const double t48 = (vT <= 6000.0) ? 1.0 : 0.0;
  const double t49 = (t48 != 0.0) ? t47 : vDUII;
  vDUII = t49;
  vUIII = 220.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_42(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.0021538001019507647;
  const double t1 = 0.04840100184082985 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.40779998898506165 + t2;
  const double t4 = vY * t3;
  const double t5 = 1.652500033378601 + t4;
  const double t6 = vY * t5;
  const double t7 = 0.3064799904823303 + t6;
  const double t8 = vY * t7;
  const double t9 = 4.439000129699707 + t8;
  vUI = t9;
  const double t10 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t11 = (t10 != 0.0) ? 24.0 : vUI;
  vUI = t11;
  const double t25 = vY * 0.001908699981868267;
  const double t26 = 0.04965599998831749 - t25;
  const double t27 = vY * t26;
  const double t28 = -0.5019999742507935 + t27;
  const double t29 = vY * t28;
  const double t30 = 2.36899995803833 + t29;
  const double t31 = vY * t30;
  const double t32 = -2.9630000591278076 + t31;
  const double t33 = vY * t32;
  const double t34 = 8.109600067138672 + t33;
  vUII = t34;
  const double t35 = (vT > 6000.0) ? 1.0 : 0.0;
  const double t36 = (t35 != 0.0) ? 17.0 : vUII;
  vUII = t36;
  vUIII = 220.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_43(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.007170000113546848 * vT;
  const double t1 = -3.0 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.007170000113546848, vUI);
  vDUI = t2;
  const double t3 = 0.004259999841451645 * vT;
  const double t4 = 3.0 + t3;
  vUII = t4;
  const double t5 = PF_DIV(0.004259999841451645, vUII);
  vDUII = t5;
  vUIII = 22.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_43(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.007170000113546848 * vT;
  const double t1 = -3.0 + t0;
  vUI = t1;
  const double t3 = 0.004259999841451645 * vT;
  const double t4 = 3.0 + t3;
  vUII = t4;
  vUIII = 22.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_44(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.0005958899855613708;
  const double t1 = 0.008790699765086174 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.04312499985098839 - t2;
  const double t4 = vY * t3;
  const double t5 = 3.8468000888824463 + t4;
  const double t6 = vY * t5;
  const double t7 = 6.916399955749512 + t6;
  vUI = t7;
  const double t8 = vY * 0.0005958899855613708;
  const double t9 = t8 * 4.0;
  const double t10 = 0.026372099295258522 - t9;
  const double t11 = vY * t10;
  const double t12 = 0.08624999970197678 - t11;
  const double t13 = vY * t12;
  const double t14 = 3.8468000888824463 + t13;
  const double t15 = 0.0010000000474974513 * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = vY * 0.000212180006201379;
  const double t18 = 0.002013999968767166 + t17;
  const double t19 = vY * t18;
  const double t20 = -0.03825699910521507 + t19;
  const double t21 = vY * t20;
  const double t22 = 1.7475999593734741 + t21;
  const double t23 = vY * t22;
  const double t24 = 7.290200233459473 + t23;
  vUII = t24;
  const double t25 = vY * 0.000212180006201379;
  const double t26 = t25 * 4.0;
  const double t27 = 0.006041999906301498 + t26;
  const double t28 = vY * t27;
  const double t29 = -0.07651399821043015 + t28;
  const double t30 = vY * t29;
  const double t31 = 1.7475999593734741 + t30;
  const double t32 = 0.0010000000474974513 * t31;
  const double t33 = PF_DIV(t32, vUII);
  vDUII = t33;
  vUIII = 30.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_44(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.0005958899855613708;
  const double t1 = 0.008790699765086174 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.04312499985098839 - t2;
  const double t4 = vY * t3;
  const double t5 = 3.8468000888824463 + t4;
  const double t6 = vY * t5;
  const double t7 = 6.916399955749512 + t6;
  vUI = t7;
  const double t17 = vY * 0.000212180006201379;
  const double t18 = 0.002013999968767166 + t17;
  const double t19 = vY * t18;
  const double t20 = -0.03825699910521507 + t19;
  const double t21 = vY * t20;
  const double t22 = 1.7475999593734741 + t21;
  const double t23 = vY * t22;
  const double t24 = 7.290200233459473 + t23;
  vUII = t24;
  vUIII = 30.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_45(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.000986000057309866 * vT;
  const double t1 = -1.75 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(0.000986000057309866, vUI);
  const double t4 = (vUI != 1.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  const double t6 = 0.00036199999158270657 * vT;
  const double t7 = 5.599999904632568 + t6;
  vUII = t7;
  const double t8 = PF_DIV(0.00036199999158270657, vUII);
  vDUII = t8;
  vUIII = 20.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_45(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.000986000057309866 * vT;
  const double t1 = -1.75 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  const double t6 = 0.00036199999158270657 * vT;
  const double t7 = 5.599999904632568 + t6;
  vUII = t7;
  vUIII = 20.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_46(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 7.88000033935532e-05 * vT;
  const double t1 = 1.5369999408721924 + t0;
  const double t2 = (2.0 > t1) ? 2.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(7.88000033935532e-05, vUI);
  const double t4 = (vUI != 2.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  const double t6 = 3.400000059627928e-05 * vT;
  const double t7 = 0.7300000190734863 + t6;
  const double t8 = (1.0 > t7) ? 1.0 : t7;
  vUII = t8;
  const double t9 = PF_DIV(3.400000059627928e-05, vUII);
  const double t10 = (vUII != 1.0) ? 1.0 : 0.0;
  const double t11 = (t10 != 0.0) ? t9 : vDUII;
  vDUII = t11;
  const double t12 = 0.00012480000441428274 * vT;
  const double t13 = 6.7729997634887695 + t12;
  vUIII = t13;
  const double t14 = PF_DIV(0.00012480000441428274, vUIII);
  vDUIII = t14;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_46(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 7.88000033935532e-05 * vT;
  const double t1 = 1.5369999408721924 + t0;
  const double t2 = (2.0 > t1) ? 2.0 : t1;
  vUI = t2;
  const double t6 = 3.400000059627928e-05 * vT;
  const double t7 = 0.7300000190734863 + t6;
  const double t8 = (1.0 > t7) ? 1.0 : t7;
  vUII = t8;
  const double t12 = 0.00012480000441428274 * vT;
  const double t13 = 6.7729997634887695 + t12;
  vUIII = t13;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_47(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 7.599999662488699e-05 * vT;
  const double t1 = 0.4300000071525574 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(7.599999662488699e-05, vUI);
  const double t4 = (vUI != 1.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  vUII = 2.0;
  vUIII = 1.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_47(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 7.599999662488699e-05 * vT;
  const double t1 = 0.4300000071525574 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  vUII = 2.0;
  vUIII = 1.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_48(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.000391999987186864 * vT;
  const double t1 = 2.1600000858306885 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.000391999987186864, vUI);
  vDUI = t2;
  vUII = 1.0;
  vUIII = 2.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_48(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.000391999987186864 * vT;
  const double t1 = 2.1600000858306885 + t0;
  vUI = t1;
  vUII = 1.0;
  vUIII = 2.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_49(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.000615999975707382 * vT;
  const double t1 = 2.140000104904175 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.000615999975707382, vUI);
  vDUI = t2;
  const double t3 = 0.00022699999681208283 * vT;
  const double t4 = 2.059999942779541 + t3;
  vUII = t4;
  const double t5 = PF_DIV(0.00022699999681208283, vUII);
  vDUII = t5;
  vUIII = 1.0499999523162842;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_49(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.000615999975707382 * vT;
  const double t1 = 2.140000104904175 + t0;
  vUI = t1;
  const double t3 = 0.00022699999681208283 * vT;
  const double t4 = 2.059999942779541 + t3;
  vUII = t4;
  vUIII = 1.0499999523162842;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_50(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.00048600000445730984 * vT;
  const double t1 = 2.3399999141693115 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.00048600000445730984, vUI);
  vDUI = t2;
  const double t3 = 0.0005360000068321824 * vT;
  const double t4 = 0.6899999976158142 + t3;
  vUII = t4;
  const double t5 = PF_DIV(0.0005360000068321824, vUII);
  vDUII = t5;
  vUIII = 3.5;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_50(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.00048600000445730984 * vT;
  const double t1 = 2.3399999141693115 + t0;
  vUI = t1;
  const double t3 = 0.0005360000068321824 * vT;
  const double t4 = 0.6899999976158142 + t3;
  vUII = t4;
  vUIII = 3.5;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_51(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0004560000088531524 * vT;
  const double t1 = 3.947999954223633 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.0004560000088531524, vUI);
  vDUI = t2;
  const double t3 = vY * 0.002427099971100688;
  const double t4 = 0.06938999891281128 - t3;
  const double t5 = vY * t4;
  const double t6 = -0.2589400112628937 + t5;
  const double t7 = vY * t6;
  const double t8 = 4.255499839782715 + t7;
  vUII = t8;
  const double t9 = vY * 0.002427099971100688;
  const double t10 = t9 * 3.0;
  const double t11 = 0.13877999782562256 - t10;
  const double t12 = vY * t11;
  const double t13 = -0.2589400112628937 + t12;
  const double t14 = 0.0010000000474974513 * t13;
  const double t15 = PF_DIV(t14, vUII);
  vDUII = t15;
  const double t16 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t17 = (t16 != 0.0) ? 7.0 : vUII;
  vUII = t17;
  vUIII = 5.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_51(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0004560000088531524 * vT;
  const double t1 = 3.947999954223633 + t0;
  vUI = t1;
  const double t3 = vY * 0.002427099971100688;
  const double t4 = 0.06938999891281128 - t3;
  const double t5 = vY * t4;
  const double t6 = -0.2589400112628937 + t5;
  const double t7 = vY * t6;
  const double t8 = 4.255499839782715 + t7;
  vUII = t8;
  const double t16 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t17 = (t16 != 0.0) ? 7.0 : vUII;
  vUII = t17;
  vUIII = 5.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_52(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 9.500000305706635e-05 * vT;
  const double t1 = 3.799999952316284 + t0;
  const double t2 = (4.0 > t1) ? 4.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(9.500000305706635e-05, vUI);
  const double t4 = (vUI != 4.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  const double t6 = 0.0003000000142492354 * vT;
  const double t7 = 4.119999885559082 + t6;
  vUII = t7;
  const double t8 = PF_DIV(0.0003000000142492354, vUII);
  vDUII = t8;
  vUIII = 7.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_52(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 9.500000305706635e-05 * vT;
  const double t1 = 3.799999952316284 + t0;
  const double t2 = (4.0 > t1) ? 4.0 : t1;
  vUI = t2;
  const double t6 = 0.0003000000142492354 * vT;
  const double t7 = 4.119999885559082 + t6;
  vUII = t7;
  vUIII = 7.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_53(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 1.0;
  const double t0 = 6.875999679323286e-05 * vT;
  const double t1 = 3.75 + t0;
  vUII = t1;
  const double t2 = PF_DIV(6.875999679323286e-05, vUII);
  vDUII = t2;
  const double t3 = 0.000232299993513152 * vT;
  const double t4 = 4.120999813079834 + t3;
  vUIII = t4;
  const double t5 = PF_DIV(0.000232299993513152, vUIII);
  vDUIII = t5;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_53(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 1.0;
  const double t0 = 6.875999679323286e-05 * vT;
  const double t1 = 3.75 + t0;
  vUII = t1;
  const double t3 = 0.000232299993513152 * vT;
  const double t4 = 4.120999813079834 + t3;
  vUIII = t4;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_54(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.00016700000560376793 * vT;
  const double t1 = 1.559999942779541 + t0;
  const double t2 = (2.0 > t1) ? 2.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(0.00016700000560376793, vUI);
  const double t4 = (vUI != 2.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  const double t6 = 0.0010400000028312206 * vT;
  const double t7 = -2.680000066757202 + t6;
  const double t8 = (vT > 4850.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t10 = PF_DIV(0.0010400000028312206, vUI);
  const double t11 = (vT > 4850.0) ? 1.0 : 0.0;
  const double t12 = (t11 != 0.0) ? t10 : vDUI;
  vDUI = t12;
  vUII = 1.0;
  const double t13 = 4.971000089426525e-05 * vT;
  const double t14 = 3.7690000534057617 + t13;
  vUIII = t14;
  const double t15 = PF_DIV(4.971000089426525e-05, vUIII);
  vDUIII = t15;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_54(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.00016700000560376793 * vT;
  const double t1 = 1.559999942779541 + t0;
  const double t2 = (2.0 > t1) ? 2.0 : t1;
  vUI = t2;
  const double t6 = 0.0010400000028312206 * vT;
  const double t7 = -2.680000066757202 + t6;
  const double t8 = (vT > 4850.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  vUII = 1.0;
  const double t13 = 4.971000089426525e-05 * vT;
  const double t14 = 3.7690000534057617 + t13;
  vUIII = t14;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_55(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0009850000496953726 * vT;
  const double t1 = -1.7999999523162842 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  const double t3 = PF_DIV(0.0009850000496953726, vUI);
  const double t4 = (vUI != 1.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  const double t6 = 0.0030799999367445707 * vT;
  const double t7 = -16.200000762939453 + t6;
  const double t8 = (vT > 6850.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t10 = PF_DIV(0.0030799999367445707, vUI);
  const double t11 = (vT > 6850.0) ? 1.0 : 0.0;
  const double t12 = (t11 != 0.0) ? t10 : vDUI;
  vDUI = t12;
  const double t13 = 0.0005939999828115106 * vT;
  const double t14 = 1.1100000143051147 + t13;
  vUII = t14;
  const double t15 = PF_DIV(0.0005939999828115106, vUII);
  vDUII = t15;
  vUIII = 1.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_55(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0009850000496953726 * vT;
  const double t1 = -1.7999999523162842 + t0;
  const double t2 = (1.0 > t1) ? 1.0 : t1;
  vUI = t2;
  const double t6 = 0.0030799999367445707 * vT;
  const double t7 = -16.200000762939453 + t6;
  const double t8 = (vT > 6850.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t13 = 0.0005939999828115106 * vT;
  const double t14 = 1.1100000143051147 + t13;
  vUII = t14;
  vUIII = 1.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_56(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0009500000160187483 * vT;
  const double t1 = 15.420000076293945 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.0009500000160187483, vUI);
  vDUI = t2;
  const double t3 = 0.003800000064074993 * vT;
  const double t4 = 1.0 + t3;
  const double t5 = (vT > 5060.0) ? 1.0 : 0.0;
  const double t6 = (t5 != 0.0) ? t4 : vUI;
  vUI = t6;
  const double t7 = PF_DIV(0.003800000064074993, vUI);
  const double t8 = (vT > 5060.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vDUI;
  vDUI = t9;
  const double t10 = 0.0035600000992417336 * vT;
  const double t11 = 13.199999809265137 + t10;
  vUII = t11;
  const double t12 = PF_DIV(0.0035600000992417336, vUII);
  vDUII = t12;
  vUIII = 12.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_56(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0009500000160187483 * vT;
  const double t1 = 15.420000076293945 + t0;
  vUI = t1;
  const double t3 = 0.003800000064074993 * vT;
  const double t4 = 1.0 + t3;
  const double t5 = (vT > 5060.0) ? 1.0 : 0.0;
  const double t6 = (t5 != 0.0) ? t4 : vUI;
  vUI = t6;
  const double t10 = 0.0035600000992417336 * vT;
  const double t11 = 13.199999809265137 + t10;
  vUII = t11;
  vUIII = 12.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_57(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.17967499792575836 * vX;
  const double t1 = 0.1196729987859726 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.983989953994751 + t2;
  const double t4 = vX * t3;
  const double t5 = 5.202902793884277 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 9.0 + t6;
  vUI = t7;
  const double t8 = 0.5390250086784363 * vX;
  const double t9 = 0.2393459975719452 + t8;
  const double t10 = vX * t9;
  const double t11 = -1.983989953994751 + t10;
  const double t12 = vDX * t11;
  vDUI = t12;
  const double t13 = vUI - 9.0;
  const double t14 = vDUI * t13;
  const double t15 = PF_DIV(t14, vUI);
  vDUI = t15;
  const double t16 = 0.05222100019454956 * vX;
  const double t17 = 0.31051498651504517 + t16;
  const double t18 = vX * t17;
  const double t19 = 1.4591959714889526 + t18;
  const double t20 = vX * t19;
  const double t21 = 5.634881973266602 - t20;
  const double t22 = PF_EXP(t21);
  const double t23 = 8.0 + t22;
  vUII = t23;
  const double t24 = 0.15666300058364868 * vX;
  const double t25 = 0.6210299730300903 + t24;
  const double t26 = vX * t25;
  const double t27 = 1.4591959714889526 + t26;
  const double t28 = vDX * t27;
  const double t29 = -t28;
  vDUII = t29;
  const double t30 = vUII - 8.0;
  const double t31 = vDUII * t30;
  const double t32 = PF_DIV(t31, vUII);
  vDUII = t32;
  const double t33 = 0.014675999991595745 * vX;
  const double t34 = 0.031860001385211945 - t33;
  const double t35 = vX * t34;
  const double t36 = 0.37240898609161377 + t35;
  const double t37 = vX * t36;
  const double t38 = 1.3409450054168701 + t37;
  const double t39 = vX * t38;
  const double t40 = 3.6291229724884033 - t39;
  const double t41 = PF_EXP(t40);
  const double t42 = 9.0 + t41;
  vUIII = t42;
  const double t43 = 0.05870399996638298 * vX;
  const double t44 = 0.09558000415563583 - t43;
  const double t45 = vX * t44;
  const double t46 = 0.7448179721832275 + t45;
  const double t47 = vX * t46;
  const double t48 = 1.3409450054168701 + t47;
  const double t49 = vDX * t48;
  const double t50 = -t49;
  vDUIII = t50;
  const double t51 = vUIII - 9.0;
  const double t52 = vDUIII * t51;
  const double t53 = PF_DIV(t52, vUIII);
  vDUIII = t53;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_57(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.17967499792575836 * vX;
  const double t1 = 0.1196729987859726 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.983989953994751 + t2;
  const double t4 = vX * t3;
  const double t5 = 5.202902793884277 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 9.0 + t6;
  vUI = t7;
  const double t16 = 0.05222100019454956 * vX;
  const double t17 = 0.31051498651504517 + t16;
  const double t18 = vX * t17;
  const double t19 = 1.4591959714889526 + t18;
  const double t20 = vX * t19;
  const double t21 = 5.634881973266602 - t20;
  const double t22 = PF_EXP(t21);
  const double t23 = 8.0 + t22;
  vUII = t23;
  const double t33 = 0.014675999991595745 * vX;
  const double t34 = 0.031860001385211945 - t33;
  const double t35 = vX * t34;
  const double t36 = 0.37240898609161377 + t35;
  const double t37 = vX * t36;
  const double t38 = 1.3409450054168701 + t37;
  const double t39 = vX * t38;
  const double t40 = 3.6291229724884033 - t39;
  const double t41 = PF_EXP(t40);
  const double t42 = 9.0 + t41;
  vUIII = t42;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_58(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.028999000787734985 * vX;
  const double t1 = 0.14949800074100494 + t0;
  const double t2 = vX * t1;
  const double t3 = 1.191467046737671 + t2;
  const double t4 = vX * t3;
  const double t5 = 4.323959827423096 - t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 9.0 + t6;
  vUII = t7;
  const double t8 = 0.08699700236320496 * vX;
  const double t9 = 0.2989960014820099 + t8;
  const double t10 = vX * t9;
  const double t11 = 1.191467046737671 + t10;
  const double t12 = vDX * t11;
  const double t13 = -t12;
  vDUII = t13;
  const double t14 = vUII - 9.0;
  const double t15 = vDUII * t14;
  const double t16 = PF_DIV(t15, vUII);
  vDUII = t16;
  vUI = vUII;
  vDUI = vDUII;
  const double t17 = 0.2779160141944885 * vX;
  const double t18 = 0.48957398533821106 + t17;
  const double t19 = vX * t18;
  const double t20 = -1.6145540475845337 + t19;
  const double t21 = vX * t20;
  const double t22 = 3.206855058670044 + t21;
  const double t23 = PF_EXP(t22);
  const double t24 = 10.0 + t23;
  vUIII = t24;
  const double t25 = 0.8337480425834656 * vX;
  const double t26 = 0.9791479706764221 + t25;
  const double t27 = vX * t26;
  const double t28 = -1.6145540475845337 + t27;
  const double t29 = vDX * t28;
  vDUIII = t29;
  const double t30 = vUIII - 10.0;
  const double t31 = vDUIII * t30;
  const double t32 = PF_DIV(t31, vUIII);
  vDUIII = t32;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_58(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.028999000787734985 * vX;
  const double t1 = 0.14949800074100494 + t0;
  const double t2 = vX * t1;
  const double t3 = 1.191467046737671 + t2;
  const double t4 = vX * t3;
  const double t5 = 4.323959827423096 - t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 9.0 + t6;
  vUII = t7;
  vUI = vUII;
  const double t17 = 0.2779160141944885 * vX;
  const double t18 = 0.48957398533821106 + t17;
  const double t19 = vX * t18;
  const double t20 = -1.6145540475845337 + t19;
  const double t21 = vX * t20;
  const double t22 = 3.206855058670044 + t21;
  const double t23 = PF_EXP(t22);
  const double t24 = 10.0 + t23;
  vUIII = t24;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_59(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.12732599675655365 * vX;
  const double t1 = 0.506659984588623 + t0;
  const double t2 = vX * t1;
  const double t3 = 0.08225800096988678 + t2;
  const double t4 = vX * t3;
  const double t5 = -2.7791759967803955 + t4;
  const double t6 = vX * t5;
  const double t7 = 4.456881999969482 + t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 9.0 + t8;
  vUI = t9;
  const double t10 = 0.5093039870262146 * vX;
  const double t11 = 1.5199799537658691 + t10;
  const double t12 = vX * t11;
  const double t13 = 0.16451600193977356 + t12;
  const double t14 = vX * t13;
  const double t15 = -2.7791759967803955 + t14;
  const double t16 = vDX * t15;
  vDUI = t16;
  const double t17 = vUI - 9.0;
  const double t18 = vDUI * t17;
  const double t19 = PF_DIV(t18, vUI);
  vDUI = t19;
  const double t20 = 0.038224998861551285 * vX;
  const double t21 = 0.26392000913619995 + t20;
  const double t22 = vX * t21;
  const double t23 = 0.1719300001859665 + t22;
  const double t24 = vX * t23;
  const double t25 = -2.0399460792541504 + t24;
  const double t26 = vX * t25;
  const double t27 = 4.689642906188965 + t26;
  const double t28 = PF_EXP(t27);
  const double t29 = 8.0 + t28;
  vUII = t29;
  const double t30 = 0.15289999544620514 * vX;
  const double t31 = 0.7917600274085999 + t30;
  const double t32 = vX * t31;
  const double t33 = 0.343860000371933 + t32;
  const double t34 = vX * t33;
  const double t35 = -2.0399460792541504 + t34;
  const double t36 = vDX * t35;
  vDUII = t36;
  const double t37 = vUII - 8.0;
  const double t38 = vDUII * t37;
  const double t39 = PF_DIV(t38, vUII);
  vDUII = t39;
  vUIII = vUII;
  vDUIII = vDUII;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_59(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.12732599675655365 * vX;
  const double t1 = 0.506659984588623 + t0;
  const double t2 = vX * t1;
  const double t3 = 0.08225800096988678 + t2;
  const double t4 = vX * t3;
  const double t5 = -2.7791759967803955 + t4;
  const double t6 = vX * t5;
  const double t7 = 4.456881999969482 + t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 9.0 + t8;
  vUI = t9;
  const double t20 = 0.038224998861551285 * vX;
  const double t21 = 0.26392000913619995 + t20;
  const double t22 = vX * t21;
  const double t23 = 0.1719300001859665 + t22;
  const double t24 = vX * t23;
  const double t25 = -2.0399460792541504 + t24;
  const double t26 = vX * t25;
  const double t27 = 4.689642906188965 + t26;
  const double t28 = PF_EXP(t27);
  const double t29 = 8.0 + t28;
  vUII = t29;
  vUIII = vUII;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_60(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 20.0;
  vUII = 25.0;
  vUIII = 100.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_60(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 20.0;
  vUII = 25.0;
  vUIII = 100.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_61(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.5662630200386047 * vX;
  const double t1 = 0.996399998664856 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.8515490293502808 + t2;
  const double t4 = vX * t3;
  const double t5 = 3.5495951175689697 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 1.0 + t6;
  vUI = t7;
  const double t8 = 1.698789119720459 * vX;
  const double t9 = 1.992799997329712 + t8;
  const double t10 = vX * t9;
  const double t11 = -1.8515490293502808 + t10;
  const double t12 = vDX * t11;
  vDUI = t12;
  const double t13 = vUI - 1.0;
  const double t14 = vDUI * t13;
  const double t15 = PF_DIV(t14, vUI);
  vDUI = t15;
  const double t16 = 0.16194400191307068 * vX;
  const double t17 = 0.35869500041007996 + t16;
  const double t18 = vX * t17;
  const double t19 = -1.4182219505310059 + t18;
  const double t20 = vX * t19;
  const double t21 = 4.052403926849365 + t20;
  const double t22 = PF_EXP(t21);
  const double t23 = 2.0 + t22;
  vUII = t23;
  const double t24 = 0.48583200573921204 * vX;
  const double t25 = 0.7173900008201599 + t24;
  const double t26 = vX * t25;
  const double t27 = -1.4182219505310059 + t26;
  const double t28 = vDX * t27;
  vDUII = t28;
  const double t29 = vUII - 2.0;
  const double t30 = vDUII * t29;
  const double t31 = PF_DIV(t30, vUII);
  vDUII = t31;
  const double t32 = 0.2510110139846802 * vX;
  const double t33 = 0.5338330268859863 + t32;
  const double t34 = vX * t33;
  const double t35 = -0.05620500072836876 + t34;
  const double t36 = vX * t35;
  const double t37 = 0.6994730234146118 + t36;
  const double t38 = vX * t37;
  const double t39 = 3.222806930541992 - t38;
  const double t40 = PF_EXP(t39);
  const double t41 = 1.0 + t40;
  vUIII = t41;
  const double t42 = 1.0040440559387207 * vX;
  const double t43 = 1.601499080657959 + t42;
  const double t44 = vX * t43;
  const double t45 = -0.11241000145673752 + t44;
  const double t46 = vX * t45;
  const double t47 = 0.6994730234146118 + t46;
  const double t48 = vDX * t47;
  const double t49 = -t48;
  vDUIII = t49;
  const double t50 = vUIII - 1.0;
  const double t51 = vDUIII * t50;
  const double t52 = PF_DIV(t51, vUIII);
  vDUIII = t52;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_61(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.5662630200386047 * vX;
  const double t1 = 0.996399998664856 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.8515490293502808 + t2;
  const double t4 = vX * t3;
  const double t5 = 3.5495951175689697 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 1.0 + t6;
  vUI = t7;
  const double t16 = 0.16194400191307068 * vX;
  const double t17 = 0.35869500041007996 + t16;
  const double t18 = vX * t17;
  const double t19 = -1.4182219505310059 + t18;
  const double t20 = vX * t19;
  const double t21 = 4.052403926849365 + t20;
  const double t22 = PF_EXP(t21);
  const double t23 = 2.0 + t22;
  vUII = t23;
  const double t32 = 0.2510110139846802 * vX;
  const double t33 = 0.5338330268859863 + t32;
  const double t34 = vX * t33;
  const double t35 = -0.05620500072836876 + t34;
  const double t36 = vX * t35;
  const double t37 = 0.6994730234146118 + t36;
  const double t38 = vX * t37;
  const double t39 = 3.222806930541992 - t38;
  const double t40 = PF_EXP(t39);
  const double t41 = 1.0 + t40;
  vUIII = t41;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_62(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.28673699498176575 * vX;
  const double t1 = 0.8277890086174011 + t0;
  const double t2 = vX * t1;
  const double t3 = 1.5408049821853638 + t2;
  const double t4 = vX * t3;
  const double t5 = 4.5336527824401855 + t4;
  const double t6 = vX * t5;
  const double t7 = 1.024374008178711 - t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 8.0 + t8;
  vUI = t9;
  const double t10 = 1.146947979927063 * vX;
  const double t11 = 2.4833669662475586 + t10;
  const double t12 = vX * t11;
  const double t13 = 3.0816099643707275 + t12;
  const double t14 = vX * t13;
  const double t15 = 4.5336527824401855 + t14;
  const double t16 = vDX * t15;
  const double t17 = -t16;
  vDUI = t17;
  const double t18 = vUI - 8.0;
  const double t19 = vDUI * t18;
  const double t20 = PF_DIV(t19, vUI);
  vDUI = t20;
  const double t21 = 0.05683999881148338 * vX;
  const double t22 = 0.37958401441574097 + t21;
  const double t23 = vX * t22;
  const double t24 = -1.5064599514007568 + t23;
  const double t25 = vX * t24;
  const double t26 = 1.9277600049972534 + t25;
  const double t27 = PF_EXP(t26);
  const double t28 = 9.0 + t27;
  vUII = t28;
  const double t29 = 0.17051999270915985 * vX;
  const double t30 = 0.7591680288314819 + t29;
  const double t31 = vX * t30;
  const double t32 = -1.5064599514007568 + t31;
  const double t33 = vDX * t32;
  vDUII = t33;
  const double t34 = vUII - 9.0;
  const double t35 = vDUII * t34;
  const double t36 = PF_DIV(t35, vUII);
  vDUII = t36;
  vUIII = 8.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_62(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.28673699498176575 * vX;
  const double t1 = 0.8277890086174011 + t0;
  const double t2 = vX * t1;
  const double t3 = 1.5408049821853638 + t2;
  const double t4 = vX * t3;
  const double t5 = 4.5336527824401855 + t4;
  const double t6 = vX * t5;
  const double t7 = 1.024374008178711 - t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 8.0 + t8;
  vUI = t9;
  const double t21 = 0.05683999881148338 * vX;
  const double t22 = 0.37958401441574097 + t21;
  const double t23 = vX * t22;
  const double t24 = -1.5064599514007568 + t23;
  const double t25 = vX * t24;
  const double t26 = 1.9277600049972534 + t25;
  const double t27 = PF_EXP(t26);
  const double t28 = 9.0 + t27;
  vUII = t28;
  vUIII = 8.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_63(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.3888449966907501 * vX;
  const double t1 = 0.8004109859466553 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.5835130214691162 + t2;
  const double t4 = vX * t3;
  const double t5 = 4.009586811065674 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 5.0 + t6;
  vUI = t7;
  const double t8 = 1.1665350198745728 * vX;
  const double t9 = 1.6008219718933105 + t8;
  const double t10 = vX * t9;
  const double t11 = -1.5835130214691162 + t10;
  const double t12 = vDX * t11;
  vDUI = t12;
  const double t13 = vUI - 5.0;
  const double t14 = vDUI * t13;
  const double t15 = PF_DIV(t14, vUI);
  vDUI = t15;
  const double t16 = 0.05547500029206276 * vX;
  const double t17 = 0.07645300030708313 + t16;
  const double t18 = vX * t17;
  const double t19 = -0.07481300085783005 + t18;
  const double t20 = vX * t19;
  const double t21 = 1.208124041557312 + t20;
  const double t22 = vX * t21;
  const double t23 = 4.362106800079346 - t22;
  const double t24 = PF_EXP(t23);
  const double t25 = 6.0 + t24;
  vUII = t25;
  const double t26 = 0.22190000116825104 * vX;
  const double t27 = 0.2293590009212494 + t26;
  const double t28 = vX * t27;
  const double t29 = -0.1496260017156601 + t28;
  const double t30 = vX * t29;
  const double t31 = 1.208124041557312 + t30;
  const double t32 = vDX * t31;
  const double t33 = -t32;
  vDUII = t33;
  const double t34 = vUII - 6.0;
  const double t35 = vDUII * t34;
  const double t36 = PF_DIV(t35, vUII);
  vDUII = t36;
  const double t37 = 0.004017000086605549 * vX;
  const double t38 = 0.04248899966478348 - t37;
  const double t39 = vX * t38;
  const double t40 = 0.5027099847793579 + t39;
  const double t41 = vX * t40;
  const double t42 = 3.4129509925842285 - t41;
  const double t43 = PF_EXP(t42);
  const double t44 = 5.0 + t43;
  vUIII = t44;
  const double t45 = 0.012051000259816647 * vX;
  const double t46 = 0.08497799932956696 - t45;
  const double t47 = vX * t46;
  const double t48 = 0.5027099847793579 + t47;
  const double t49 = vDX * t48;
  const double t50 = -t49;
  vDUIII = t50;
  const double t51 = vUIII - 5.0;
  const double t52 = vDUIII * t51;
  const double t53 = PF_DIV(t52, vUIII);
  vDUIII = t53;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_63(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.3888449966907501 * vX;
  const double t1 = 0.8004109859466553 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.5835130214691162 + t2;
  const double t4 = vX * t3;
  const double t5 = 4.009586811065674 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 5.0 + t6;
  vUI = t7;
  const double t16 = 0.05547500029206276 * vX;
  const double t17 = 0.07645300030708313 + t16;
  const double t18 = vX * t17;
  const double t19 = -0.07481300085783005 + t18;
  const double t20 = vX * t19;
  const double t21 = 1.208124041557312 + t20;
  const double t22 = vX * t21;
  const double t23 = 4.362106800079346 - t22;
  const double t24 = PF_EXP(t23);
  const double t25 = 6.0 + t24;
  vUII = t25;
  const double t37 = 0.004017000086605549 * vX;
  const double t38 = 0.04248899966478348 - t37;
  const double t39 = vX * t38;
  const double t40 = 0.5027099847793579 + t39;
  const double t41 = vX * t40;
  const double t42 = 3.4129509925842285 - t41;
  const double t43 = PF_EXP(t42);
  const double t44 = 5.0 + t43;
  vUIII = t44;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_64(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.24020299315452576 * vX;
  const double t1 = 0.5700939893722534 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.2493549585342407 + t2;
  const double t4 = vX * t3;
  const double t5 = 4.791660785675049 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 16.0 + t6;
  vUI = t7;
  const double t8 = 0.7206089496612549 * vX;
  const double t9 = 1.1401879787445068 + t8;
  const double t10 = vX * t9;
  const double t11 = -1.2493549585342407 + t10;
  const double t12 = vDX * t11;
  vDUI = t12;
  const double t13 = vUI - 16.0;
  const double t14 = vDUI * t13;
  const double t15 = PF_DIV(t14, vUI);
  vDUI = t15;
  const double t16 = 0.131631001830101 * vX;
  const double t17 = 0.005880000069737434 + t16;
  const double t18 = vX * t17;
  const double t19 = 0.2959649860858917 + t18;
  const double t20 = vX * t19;
  const double t21 = 4.472548961639404 - t20;
  const double t22 = PF_EXP(t21);
  const double t23 = 15.0 + t22;
  vUII = t23;
  const double t24 = 0.39489299058914185 * vX;
  const double t25 = 0.011760000139474869 + t24;
  const double t26 = vX * t25;
  const double t27 = 0.2959649860858917 + t26;
  const double t28 = vDX * t27;
  const double t29 = -t28;
  vDUII = t29;
  const double t30 = vUII - 15.0;
  const double t31 = vDUII * t30;
  const double t32 = PF_DIV(t31, vUII);
  vDUII = t32;
  vUIII = vUII;
  vDUIII = vDUII;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_64(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.24020299315452576 * vX;
  const double t1 = 0.5700939893722534 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.2493549585342407 + t2;
  const double t4 = vX * t3;
  const double t5 = 4.791660785675049 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 16.0 + t6;
  vUI = t7;
  const double t16 = 0.131631001830101 * vX;
  const double t17 = 0.005880000069737434 + t16;
  const double t18 = vX * t17;
  const double t19 = 0.2959649860858917 + t18;
  const double t20 = vX * t19;
  const double t21 = 4.472548961639404 - t20;
  const double t22 = PF_EXP(t21);
  const double t23 = 15.0 + t22;
  vUII = t23;
  vUIII = vUII;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_65(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.21621400117874146 * vX;
  const double t1 = 0.08667100220918655 - t0;
  const double t2 = vX * t1;
  const double t3 = 3.1210360527038574 + t2;
  const double t4 = vX * t3;
  const double t5 = 3.0296459197998047 - t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 17.0 + t6;
  vUI = t7;
  const double t8 = 0.6486420035362244 * vX;
  const double t9 = 0.1733420044183731 - t8;
  const double t10 = vX * t9;
  const double t11 = 3.1210360527038574 + t10;
  const double t12 = vDX * t11;
  const double t13 = -t12;
  vDUI = t13;
  const double t14 = vUI - 17.0;
  const double t15 = vDUI * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = 0.3035750091075897 * vX;
  const double t18 = 0.43144699931144714 + t17;
  const double t19 = vX * t18;
  const double t20 = -0.38226500153541565 + t19;
  const double t21 = vX * t20;
  const double t22 = 1.2706199884414673 + t21;
  const double t23 = vX * t22;
  const double t24 = 3.465322971343994 - t23;
  const double t25 = PF_EXP(t24);
  const double t26 = 18.0 + t25;
  vUII = t26;
  const double t27 = 1.2143000364303589 * vX;
  const double t28 = 1.294340968132019 + t27;
  const double t29 = vX * t28;
  const double t30 = -0.7645300030708313 + t29;
  const double t31 = vX * t30;
  const double t32 = 1.2706199884414673 + t31;
  const double t33 = vDX * t32;
  const double t34 = -t33;
  vDUII = t34;
  const double t35 = vUII - 18.0;
  const double t36 = vDUII * t35;
  const double t37 = PF_DIV(t36, vUII);
  vDUII = t37;
  vUIII = vUII;
  vDUIII = vDUII;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_65(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.21621400117874146 * vX;
  const double t1 = 0.08667100220918655 - t0;
  const double t2 = vX * t1;
  const double t3 = 3.1210360527038574 + t2;
  const double t4 = vX * t3;
  const double t5 = 3.0296459197998047 - t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 17.0 + t6;
  vUI = t7;
  const double t17 = 0.3035750091075897 * vX;
  const double t18 = 0.43144699931144714 + t17;
  const double t19 = vX * t18;
  const double t20 = -0.38226500153541565 + t19;
  const double t21 = vX * t20;
  const double t22 = 1.2706199884414673 + t21;
  const double t23 = vX * t22;
  const double t24 = 3.465322971343994 - t23;
  const double t25 = PF_EXP(t24);
  const double t26 = 18.0 + t25;
  vUII = t26;
  vUIII = vUII;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_66(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.07119599729776382 * vX;
  const double t1 = 0.1331389993429184 - t0;
  const double t2 = vX * t1;
  const double t3 = 2.3739259243011475 + t2;
  const double t4 = vX * t3;
  const double t5 = 1.610084056854248 - t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 16.0 + t6;
  vUIII = t7;
  const double t8 = 0.21358799934387207 * vX;
  const double t9 = 0.2662779986858368 - t8;
  const double t10 = vX * t9;
  const double t11 = 2.3739259243011475 + t10;
  const double t12 = vDX * t11;
  const double t13 = -t12;
  vDUIII = t13;
  const double t14 = vUIII - 16.0;
  const double t15 = vDUIII * t14;
  const double t16 = PF_DIV(t15, vUIII);
  vDUIII = t16;
  vUI = vUIII;
  vDUI = vDUIII;
  vUII = vUIII;
  vDUII = vDUIII;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_66(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.07119599729776382 * vX;
  const double t1 = 0.1331389993429184 - t0;
  const double t2 = vX * t1;
  const double t3 = 2.3739259243011475 + t2;
  const double t4 = vX * t3;
  const double t5 = 1.610084056854248 - t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 16.0 + t6;
  vUIII = t7;
  vUI = vUIII;
  vUII = vUIII;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_67(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.09581299871206284 * vX;
  const double t1 = 0.21526700258255005 + t0;
  const double t2 = vX * t1;
  const double t3 = 0.5615149736404419 + t2;
  const double t4 = vX * t3;
  const double t5 = 2.9686028957366943 + t4;
  const double t6 = vX * t5;
  const double t7 = 2.8956480026245117 - t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 13.0 + t8;
  vUI = t9;
  const double t10 = 0.38325199484825134 * vX;
  const double t11 = 0.6458010077476501 + t10;
  const double t12 = vX * t11;
  const double t13 = 1.1230299472808838 + t12;
  const double t14 = vX * t13;
  const double t15 = 2.9686028957366943 + t14;
  const double t16 = vDX * t15;
  const double t17 = -t16;
  vDUI = t17;
  const double t18 = vUI - 13.0;
  const double t19 = vDUI * t18;
  const double t20 = PF_DIV(t19, vUI);
  vDUI = t20;
  const double t21 = 0.18604199588298798 * vX;
  const double t22 = 0.34373798966407776 + t21;
  const double t23 = vX * t22;
  const double t24 = -0.22662200033664703 + t23;
  const double t25 = vX * t24;
  const double t26 = 0.8522089719772339 + t25;
  const double t27 = vX * t26;
  const double t28 = 3.2025420665740967 - t27;
  const double t29 = PF_EXP(t28);
  const double t30 = 14.0 + t29;
  vUII = t30;
  const double t31 = 0.7441679835319519 * vX;
  const double t32 = 1.0312139987945557 + t31;
  const double t33 = vX * t32;
  const double t34 = -0.45324400067329407 + t33;
  const double t35 = vX * t34;
  const double t36 = 0.8522089719772339 + t35;
  const double t37 = vDX * t36;
  const double t38 = -t37;
  vDUII = t38;
  const double t39 = vUII - 14.0;
  const double t40 = vDUII * t39;
  const double t41 = PF_DIV(t40, vUII);
  vDUII = t41;
  vUIII = vUII;
  vDUIII = vDUII;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_67(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.09581299871206284 * vX;
  const double t1 = 0.21526700258255005 + t0;
  const double t2 = vX * t1;
  const double t3 = 0.5615149736404419 + t2;
  const double t4 = vX * t3;
  const double t5 = 2.9686028957366943 + t4;
  const double t6 = vX * t5;
  const double t7 = 2.8956480026245117 - t6;
  const double t8 = PF_EXP(t7);
  const double t9 = 13.0 + t8;
  vUI = t9;
  const double t21 = 0.18604199588298798 * vX;
  const double t22 = 0.34373798966407776 + t21;
  const double t23 = vX * t22;
  const double t24 = -0.22662200033664703 + t23;
  const double t25 = vX * t24;
  const double t26 = 0.8522089719772339 + t25;
  const double t27 = vX * t26;
  const double t28 = 3.2025420665740967 - t27;
  const double t29 = PF_EXP(t28);
  const double t30 = 14.0 + t29;
  vUII = t30;
  vUIII = vUII;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_68(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.034811001271009445 * vX;
  const double t1 = 1.0816030502319336 + t0;
  const double t2 = vX * t1;
  const double t3 = 4.947569847106934 + t2;
  const double t4 = vX * t3;
  const double t5 = 1.021172046661377 - t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 8.0 + t6;
  vUI = t7;
  const double t8 = 0.10443300008773804 * vX;
  const double t9 = 2.163206100463867 + t8;
  const double t10 = vX * t9;
  const double t11 = 4.947569847106934 + t10;
  const double t12 = vDX * t11;
  const double t13 = -t12;
  vDUI = t13;
  const double t14 = vUI - 8.0;
  const double t15 = vDUI * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = 0.8133029937744141 * vX;
  const double t18 = 1.9403949975967407 + t17;
  const double t19 = vX * t18;
  const double t20 = -1.2953269481658936 + t19;
  const double t21 = vX * t20;
  const double t22 = 2.173151969909668 + t21;
  const double t23 = PF_EXP(t22);
  const double t24 = 9.0 + t23;
  vUII = t24;
  const double t25 = 2.439908981323242 * vX;
  const double t26 = 3.8807899951934814 + t25;
  const double t27 = vX * t26;
  const double t28 = -1.2953269481658936 + t27;
  const double t29 = vDX * t28;
  vDUII = t29;
  const double t30 = vUII - 9.0;
  const double t31 = vDUII * t30;
  const double t32 = PF_DIV(t31, vUII);
  vDUII = t32;
  const double t33 = 0.5543969869613647 * vX;
  const double t34 = 0.7999110221862793 + t33;
  const double t35 = vX * t34;
  const double t36 = -3.383368968963623 + t35;
  const double t37 = vX * t36;
  const double t38 = -0.5673980116844177 + t37;
  const double t39 = PF_EXP(t38);
  const double t40 = 8.0 + t39;
  vUIII = t40;
  const double t41 = 1.6631909608840942 * vX;
  const double t42 = 1.5998220443725586 + t41;
  const double t43 = vX * t42;
  const double t44 = -3.383368968963623 + t43;
  const double t45 = vDX * t44;
  vDUIII = t45;
  const double t46 = vUIII - 8.0;
  const double t47 = vDUIII * t46;
  const double t48 = PF_DIV(t47, vUIII);
  vDUIII = t48;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_68(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.034811001271009445 * vX;
  const double t1 = 1.0816030502319336 + t0;
  const double t2 = vX * t1;
  const double t3 = 4.947569847106934 + t2;
  const double t4 = vX * t3;
  const double t5 = 1.021172046661377 - t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 8.0 + t6;
  vUI = t7;
  const double t17 = 0.8133029937744141 * vX;
  const double t18 = 1.9403949975967407 + t17;
  const double t19 = vX * t18;
  const double t20 = -1.2953269481658936 + t19;
  const double t21 = vX * t20;
  const double t22 = 2.173151969909668 + t21;
  const double t23 = PF_EXP(t22);
  const double t24 = 9.0 + t23;
  vUII = t24;
  const double t33 = 0.5543969869613647 * vX;
  const double t34 = 0.7999110221862793 + t33;
  const double t35 = vX * t34;
  const double t36 = -3.383368968963623 + t35;
  const double t37 = vX * t36;
  const double t38 = -0.5673980116844177 + t37;
  const double t39 = PF_EXP(t38);
  const double t40 = 8.0 + t39;
  vUIII = t40;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_69(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.2692370116710663 * vX;
  const double t1 = 1.938689947128296 + t0;
  const double t2 = vX * t1;
  const double t3 = 6.688837051391602 + t2;
  const double t4 = vX * t3;
  const double t5 = -2.3505489826202393 - t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 1.0 + t6;
  vUI = t7;
  const double t8 = 0.8077110052108765 * vX;
  const double t9 = 3.877379894256592 + t8;
  const double t10 = vX * t9;
  const double t11 = 6.688837051391602 + t10;
  const double t12 = vDX * t11;
  const double t13 = -t12;
  vDUI = t13;
  const double t14 = vUI - 1.0;
  const double t15 = vDUI * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = 0.44756999611854553 * vX;
  const double t18 = 2.35526704788208 + t17;
  const double t19 = vX * t18;
  const double t20 = 7.390443801879883 + t19;
  const double t21 = vX * t20;
  const double t22 = -3.0474650859832764 - t21;
  const double t23 = PF_EXP(t22);
  const double t24 = 2.0 + t23;
  vUII = t24;
  const double t25 = 1.342710018157959 * vX;
  const double t26 = 4.71053409576416 + t25;
  const double t27 = vX * t26;
  const double t28 = 7.390443801879883 + t27;
  const double t29 = vDX * t28;
  const double t30 = -t29;
  vDUII = t30;
  const double t31 = vUII - 2.0;
  const double t32 = vDUII * t31;
  const double t33 = PF_DIV(t32, vUII);
  vDUII = t33;
  const double t34 = 0.9401710033416748 * vX;
  const double t35 = 4.579384803771973 + t34;
  const double t36 = vX * t35;
  const double t37 = 10.560551643371582 + t36;
  const double t38 = vX * t37;
  const double t39 = -6.192056179046631 - t38;
  const double t40 = PF_EXP(t39);
  const double t41 = 1.0 + t40;
  vUIII = t41;
  const double t42 = 2.8205130100250244 * vX;
  const double t43 = 9.158769607543945 + t42;
  const double t44 = vX * t43;
  const double t45 = 10.560551643371582 + t44;
  const double t46 = vDX * t45;
  const double t47 = -t46;
  vDUIII = t47;
  const double t48 = vUIII - 1.0;
  const double t49 = vDUIII * t48;
  const double t50 = PF_DIV(t49, vUIII);
  vDUIII = t50;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_69(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.2692370116710663 * vX;
  const double t1 = 1.938689947128296 + t0;
  const double t2 = vX * t1;
  const double t3 = 6.688837051391602 + t2;
  const double t4 = vX * t3;
  const double t5 = -2.3505489826202393 - t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 1.0 + t6;
  vUI = t7;
  const double t17 = 0.44756999611854553 * vX;
  const double t18 = 2.35526704788208 + t17;
  const double t19 = vX * t18;
  const double t20 = 7.390443801879883 + t19;
  const double t21 = vX * t20;
  const double t22 = -3.0474650859832764 - t21;
  const double t23 = PF_EXP(t22);
  const double t24 = 2.0 + t23;
  vUII = t24;
  const double t34 = 0.9401710033416748 * vX;
  const double t35 = 4.579384803771973 + t34;
  const double t36 = vX * t35;
  const double t37 = 10.560551643371582 + t36;
  const double t38 = vX * t37;
  const double t39 = -6.192056179046631 - t38;
  const double t40 = PF_EXP(t39);
  const double t41 = 1.0 + t40;
  vUIII = t41;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_70(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.19336199760437012 * vX;
  const double t1 = 0.6085360050201416 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.1402640342712402 + t2;
  const double t4 = vX * t3;
  const double t5 = 1.537093997001648 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 4.0 + t6;
  vUI = t7;
  const double t8 = 0.5800859928131104 * vX;
  const double t9 = 1.2170720100402832 + t8;
  const double t10 = vX * t9;
  const double t11 = -1.1402640342712402 + t10;
  const double t12 = vDX * t11;
  vDUI = t12;
  const double t13 = vUI - 4.0;
  const double t14 = vDUI * t13;
  const double t15 = PF_DIV(t14, vUI);
  vDUI = t15;
  const double t16 = 0.00015199999324977398 * vT;
  const double t17 = 0.6600000262260437 + t16;
  const double t18 = (1.0 > t17) ? 1.0 : t17;
  vUII = t18;
  const double t19 = PF_DIV(0.00015199999324977398, vUII);
  const double t20 = (vUII != 1.0) ? 1.0 : 0.0;
  const double t21 = (t20 != 0.0) ? t19 : vDUII;
  vDUII = t21;
  const double t22 = 0.00048600000445730984 * vT;
  const double t23 = -1.090000033378601 + t22;
  const double t24 = (vT > 5250.0) ? 1.0 : 0.0;
  const double t25 = (t24 != 0.0) ? t23 : vUII;
  vUII = t25;
  const double t26 = PF_DIV(0.00048600000445730984, vUII);
  const double t27 = (vT > 5250.0) ? 1.0 : 0.0;
  const double t28 = (t27 != 0.0) ? t26 : vDUII;
  vDUII = t28;
  vUIII = 5.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_70(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.19336199760437012 * vX;
  const double t1 = 0.6085360050201416 + t0;
  const double t2 = vX * t1;
  const double t3 = -1.1402640342712402 + t2;
  const double t4 = vX * t3;
  const double t5 = 1.537093997001648 + t4;
  const double t6 = PF_EXP(t5);
  const double t7 = 4.0 + t6;
  vUI = t7;
  const double t16 = 0.00015199999324977398 * vT;
  const double t17 = 0.6600000262260437 + t16;
  const double t18 = (1.0 > t17) ? 1.0 : t17;
  vUII = t18;
  const double t22 = 0.00048600000445730984 * vT;
  const double t23 = -1.090000033378601 + t22;
  const double t24 = (vT > 5250.0) ? 1.0 : 0.0;
  const double t25 = (t24 != 0.0) ? t23 : vUII;
  vUII = t25;
  vUIII = 5.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_71(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.003684799885377288;
  const double t1 = 0.07288700342178345 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.5786200165748596 - t2;
  const double t4 = vY * t3;
  const double t5 = 0.40700000524520874 + t4;
  const double t6 = vY * t5;
  const double t7 = 4.17579984664917 + t6;
  vUI = t7;
  const double t8 = vY * 0.003684799885377288;
  const double t9 = t8 * 4.0;
  const double t10 = 0.21866101026535034 - t9;
  const double t11 = vY * t10;
  const double t12 = 1.1572400331497192 - t11;
  const double t13 = vY * t12;
  const double t14 = 0.40700000524520874 + t13;
  const double t15 = 0.0010000000474974513 * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = 0.0030950000509619713 * vT;
  const double t18 = -2.9790000915527344 + t17;
  vUII = t18;
  const double t19 = PF_DIV(0.0030950000509619713, vUII);
  vDUII = t19;
  vUIII = 30.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_71(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.003684799885377288;
  const double t1 = 0.07288700342178345 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.5786200165748596 - t2;
  const double t4 = vY * t3;
  const double t5 = 0.40700000524520874 + t4;
  const double t6 = vY * t5;
  const double t7 = 4.17579984664917 + t6;
  vUI = t7;
  const double t17 = 0.0030950000509619713 * vT;
  const double t18 = -2.9790000915527344 + t17;
  vUII = t18;
  vUIII = 30.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_72(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.0003073900006711483;
  const double t1 = 0.0074860998429358006 + t0;
  const double t2 = vY * t1;
  const double t3 = 0.34935998916625977 + t2;
  const double t4 = vY * t3;
  const double t5 = 0.8177599906921387 + t4;
  const double t6 = vY * t5;
  const double t7 = 3.0678999423980713 + t6;
  vUI = t7;
  const double t8 = vY * 0.0003073900006711483;
  const double t9 = t8 * 4.0;
  const double t10 = 0.02245829999446869 + t9;
  const double t11 = vY * t10;
  const double t12 = 0.6987199783325195 + t11;
  const double t13 = vY * t12;
  const double t14 = 0.8177599906921387 + t13;
  const double t15 = 0.0010000000474974513 * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = vY * 0.00089565000962466;
  const double t18 = 0.031036000698804855 - t17;
  const double t19 = vY * t18;
  const double t20 = 0.5644299983978271 - t19;
  const double t21 = vY * t20;
  const double t22 = 2.0102999210357666 + t21;
  const double t23 = vY * t22;
  const double t24 = 1.68340003490448 + t23;
  vUII = t24;
  const double t25 = vY * 0.00089565000962466;
  const double t26 = t25 * 4.0;
  const double t27 = 0.09310799837112427 - t26;
  const double t28 = vY * t27;
  const double t29 = 1.1288599967956543 - t28;
  const double t30 = vY * t29;
  const double t31 = 2.0102999210357666 + t30;
  const double t32 = 0.0010000000474974513 * t31;
  const double t33 = PF_DIV(t32, vUII);
  vDUII = t33;
  vUIII = 15.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_72(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.0003073900006711483;
  const double t1 = 0.0074860998429358006 + t0;
  const double t2 = vY * t1;
  const double t3 = 0.34935998916625977 + t2;
  const double t4 = vY * t3;
  const double t5 = 0.8177599906921387 + t4;
  const double t6 = vY * t5;
  const double t7 = 3.0678999423980713 + t6;
  vUI = t7;
  const double t17 = vY * 0.00089565000962466;
  const double t18 = 0.031036000698804855 - t17;
  const double t19 = vY * t18;
  const double t20 = 0.5644299983978271 - t19;
  const double t21 = vY * t20;
  const double t22 = 2.0102999210357666 + t21;
  const double t23 = vY * t22;
  const double t24 = 1.68340003490448 + t23;
  vUII = t24;
  vUIII = 15.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_73(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.0018400000408291817;
  const double t1 = 0.04192399978637695 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.34373000264167786 + t2;
  const double t4 = vY * t3;
  const double t5 = 1.4433000087738037 + t4;
  const double t6 = vY * t5;
  const double t7 = -0.25056999921798706 + t6;
  const double t8 = vY * t7;
  const double t9 = 0.3950999975204468 + t8;
  vUI = t9;
  const double t10 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t11 = (t10 != 0.0) ? 23.0 : vUI;
  vUI = t11;
  const double t12 = vY * 0.0018400000408291817;
  const double t13 = t12 * 5.0;
  const double t14 = 0.1676959991455078 - t13;
  const double t15 = vY * t14;
  const double t16 = -1.031190037727356 + t15;
  const double t17 = vY * t16;
  const double t18 = 2.8866000175476074 + t17;
  const double t19 = vY * t18;
  const double t20 = -0.25056999921798706 + t19;
  const double t21 = 0.0010000000474974513 * t20;
  const double t22 = PF_DIV(t21, vUI);
  const double t23 = (vT <= 12000.0) ? 1.0 : 0.0;
  const double t24 = (t23 != 0.0) ? t22 : vDUI;
  vDUI = t24;
  const double t25 = vY * 0.000557939987629652;
  const double t26 = 0.008497100323438644 - t25;
  const double t27 = vY * t26;
  const double t28 = 0.3303000032901764 - t27;
  const double t29 = vY * t28;
  const double t30 = 1.0396000146865845 + t29;
  const double t31 = vY * t30;
  const double t32 = 1.0549999475479126 + t31;
  vUII = t32;
  const double t33 = vY * 0.000557939987629652;
  const double t34 = t33 * 4.0;
  const double t35 = 0.025491300970315933 - t34;
  const double t36 = vY * t35;
  const double t37 = 0.6606000065803528 - t36;
  const double t38 = vY * t37;
  const double t39 = 1.0396000146865845 + t38;
  const double t40 = 0.0010000000474974513 * t39;
  const double t41 = PF_DIV(t40, vUII);
  vDUII = t41;
  vUIII = 20.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_73(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.0018400000408291817;
  const double t1 = 0.04192399978637695 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.34373000264167786 + t2;
  const double t4 = vY * t3;
  const double t5 = 1.4433000087738037 + t4;
  const double t6 = vY * t5;
  const double t7 = -0.25056999921798706 + t6;
  const double t8 = vY * t7;
  const double t9 = 0.3950999975204468 + t8;
  vUI = t9;
  const double t10 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t11 = (t10 != 0.0) ? 23.0 : vUI;
  vUI = t11;
  const double t25 = vY * 0.000557939987629652;
  const double t26 = 0.008497100323438644 - t25;
  const double t27 = vY * t26;
  const double t28 = 0.3303000032901764 - t27;
  const double t29 = vY * t28;
  const double t30 = 1.0396000146865845 + t29;
  const double t31 = vY * t30;
  const double t32 = 1.0549999475479126 + t31;
  vUII = t32;
  vUIII = 20.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_74(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.003933100029826164;
  const double t1 = 0.09075000137090683 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.420960009098053 + t2;
  const double t4 = vY * t3;
  const double t5 = 0.7272099852561951 + t4;
  const double t6 = vY * t5;
  const double t7 = 5.5671000480651855 + t6;
  vUI = t7;
  const double t8 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? 29.0 : vUI;
  vUI = t9;
  const double t10 = vY * 0.003933100029826164;
  const double t11 = t10 * 4.0;
  const double t12 = 0.2722499966621399 - t11;
  const double t13 = vY * t12;
  const double t14 = -0.841920018196106 + t13;
  const double t15 = vY * t14;
  const double t16 = 0.7272099852561951 + t15;
  const double t17 = 0.0010000000474974513 * t16;
  const double t18 = PF_DIV(t17, vUI);
  const double t19 = (vT <= 12000.0) ? 1.0 : 0.0;
  const double t20 = (t19 != 0.0) ? t18 : vDUI;
  vDUI = t20;
  const double t21 = vY * 0.0018544000340625644;
  const double t22 = 0.05072399973869324 - t21;
  const double t23 = vY * t22;
  const double t24 = -0.2853200137615204 + t23;
  const double t25 = vY * t24;
  const double t26 = 0.5999900102615356 + t25;
  const double t27 = vY * t26;
  const double t28 = 6.569900035858154 + t27;
  vUII = t28;
  const double t29 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t30 = (t29 != 0.0) ? 22.0 : vUII;
  vUII = t30;
  const double t31 = vY * 0.0018544000340625644;
  const double t32 = t31 * 4.0;
  const double t33 = 0.1521719992160797 - t32;
  const double t34 = vY * t33;
  const double t35 = -0.5706400275230408 + t34;
  const double t36 = vY * t35;
  const double t37 = 0.5999900102615356 + t36;
  const double t38 = 0.0010000000474974513 * t37;
  const double t39 = PF_DIV(t38, vUII);
  const double t40 = (vT <= 12000.0) ? 1.0 : 0.0;
  const double t41 = (t40 != 0.0) ? t39 : vDUII;
  vDUII = t41;
  vUIII = 20.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_74(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.003933100029826164;
  const double t1 = 0.09075000137090683 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.420960009098053 + t2;
  const double t4 = vY * t3;
  const double t5 = 0.7272099852561951 + t4;
  const double t6 = vY * t5;
  const double t7 = 5.5671000480651855 + t6;
  vUI = t7;
  const double t8 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? 29.0 : vUI;
  vUI = t9;
  const double t21 = vY * 0.0018544000340625644;
  const double t22 = 0.05072399973869324 - t21;
  const double t23 = vY * t22;
  const double t24 = -0.2853200137615204 + t23;
  const double t25 = vY * t24;
  const double t26 = 0.5999900102615356 + t25;
  const double t27 = vY * t26;
  const double t28 = 6.569900035858154 + t27;
  vUII = t28;
  const double t29 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t30 = (t29 != 0.0) ? 22.0 : vUII;
  vUII = t30;
  vUIII = 20.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_75(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = vY * 0.0019974999595433474;
  const double t1 = 0.044252000749111176 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.6818100214004517 - t2;
  const double t4 = vY * t3;
  const double t5 = -0.3251599967479706 + t4;
  const double t6 = vY * t5;
  const double t7 = 8.664299964904785 + t6;
  vUI = t7;
  const double t8 = vY * 0.0019974999595433474;
  const double t9 = t8 * 4.0;
  const double t10 = 0.13275599479675293 - t9;
  const double t11 = vY * t10;
  const double t12 = 1.3636200428009033 - t11;
  const double t13 = vY * t12;
  const double t14 = -0.3251599967479706 + t13;
  const double t15 = 0.0010000000474974513 * t14;
  const double t16 = PF_DIV(t15, vUI);
  vDUI = t16;
  const double t17 = vY * 0.0028792000375688076;
  const double t18 = 0.06498400121927261 - t17;
  const double t19 = vY * t18;
  const double t20 = 0.6529200077056885 - t19;
  const double t21 = vY * t20;
  const double t22 = -0.3813999891281128 + t21;
  const double t23 = vY * t22;
  const double t24 = 9.708600044250488 + t23;
  vUII = t24;
  const double t25 = vY * 0.0028792000375688076;
  const double t26 = t25 * 4.0;
  const double t27 = 0.19495201110839844 - t26;
  const double t28 = vY * t27;
  const double t29 = 1.305840015411377 - t28;
  const double t30 = vY * t29;
  const double t31 = -0.3813999891281128 + t30;
  const double t32 = 0.0010000000474974513 * t31;
  const double t33 = PF_DIV(t32, vUII);
  vDUII = t33;
  vUIII = 10.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_75(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = vY * 0.0019974999595433474;
  const double t1 = 0.044252000749111176 - t0;
  const double t2 = vY * t1;
  const double t3 = 0.6818100214004517 - t2;
  const double t4 = vY * t3;
  const double t5 = -0.3251599967479706 + t4;
  const double t6 = vY * t5;
  const double t7 = 8.664299964904785 + t6;
  vUI = t7;
  const double t17 = vY * 0.0028792000375688076;
  const double t18 = 0.06498400121927261 - t17;
  const double t19 = vY * t18;
  const double t20 = 0.6529200077056885 - t19;
  const double t21 = vY * t20;
  const double t22 = -0.3813999891281128 + t21;
  const double t23 = vY * t22;
  const double t24 = 9.708600044250488 + t23;
  vUII = t24;
  vUIII = 10.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_76(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0013376000570133328 * vY;
  const double t1 = 0.033511001616716385 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.3438900113105774 + t2;
  const double t4 = vY * t3;
  const double t5 = 1.9387999773025513 + t4;
  const double t6 = vY * t5;
  const double t7 = -2.4119999408721924 + t6;
  const double t8 = vY * t7;
  const double t9 = 11.069999694824219 + t8;
  vUI = t9;
  const double t10 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t11 = (t10 != 0.0) ? 30.0 : vUI;
  vUI = t11;
  const double t12 = 0.006688000168651342 * vY;
  const double t13 = 0.13404400646686554 - t12;
  const double t14 = vY * t13;
  const double t15 = -1.031670093536377 + t14;
  const double t16 = vY * t15;
  const double t17 = 3.8775999546051025 + t16;
  const double t18 = vY * t17;
  const double t19 = -2.4119999408721924 + t18;
  const double t20 = 0.0010000000474974513 * t19;
  const double t21 = PF_DIV(t20, vUI);
  const double t22 = (vT <= 12000.0) ? 1.0 : 0.0;
  const double t23 = (t22 != 0.0) ? t21 : vDUI;
  vDUI = t23;
  vUII = 15.0;
  vUIII = 20.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_76(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0013376000570133328 * vY;
  const double t1 = 0.033511001616716385 - t0;
  const double t2 = vY * t1;
  const double t3 = -0.3438900113105774 + t2;
  const double t4 = vY * t3;
  const double t5 = 1.9387999773025513 + t4;
  const double t6 = vY * t5;
  const double t7 = -2.4119999408721924 + t6;
  const double t8 = vY * t7;
  const double t9 = 11.069999694824219 + t8;
  vUI = t9;
  const double t10 = (vT > 12000.0) ? 1.0 : 0.0;
  const double t11 = (t10 != 0.0) ? 30.0 : vUI;
  vUI = t11;
  vUII = 15.0;
  vUIII = 20.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_77(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0012700000079348683 * vT;
  const double t1 = 16.399999618530273 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.0012700000079348683, vUI);
  vDUI = t2;
  const double t3 = 0.0026877999771386385 * vY;
  const double t4 = 0.061218999326229095 - t3;
  const double t5 = vY * t4;
  const double t6 = 0.5723400115966797 - t5;
  const double t7 = vY * t6;
  const double t8 = -1.0362999439239502 + t7;
  const double t9 = vY * t8;
  const double t10 = 6.571199893951416 + t9;
  vUII = t10;
  const double t11 = vY * 4.0;
  const double t12 = t11 * 0.0026877999771386385;
  const double t13 = 0.1836569905281067 - t12;
  const double t14 = vY * t13;
  const double t15 = 1.1446800231933594 - t14;
  const double t16 = vY * t15;
  const double t17 = -1.0362999439239502 + t16;
  const double t18 = 0.0010000000474974513 * t17;
  vDUII = t18;
  const double t19 = PF_DIV(vDUII, vUII);
  vDUII = t19;
  vUIII = 15.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_77(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0012700000079348683 * vT;
  const double t1 = 16.399999618530273 + t0;
  vUI = t1;
  const double t3 = 0.0026877999771386385 * vY;
  const double t4 = 0.061218999326229095 - t3;
  const double t5 = vY * t4;
  const double t6 = 0.5723400115966797 - t5;
  const double t7 = vY * t6;
  const double t8 = -1.0362999439239502 + t7;
  const double t9 = vY * t8;
  const double t10 = 6.571199893951416 + t9;
  vUII = t10;
  vUIII = 15.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_78(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0002789999998640269 * vT;
  const double t1 = 1.2400000095367432 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.0002789999998640269, vUI);
  vDUI = t2;
  const double t3 = vY * 0.0016586000565439463;
  const double t4 = 0.0028438998851925135 + t3;
  const double t5 = vY * t4;
  const double t6 = -0.04080900177359581 + t5;
  const double t7 = vY * t6;
  const double t8 = 1.0546000003814697 + t7;
  vUII = t8;
  const double t9 = vY * 0.0016586000565439463;
  const double t10 = t9 * 3.0;
  const double t11 = 0.005687799770385027 + t10;
  const double t12 = vY * t11;
  const double t13 = -0.04080900177359581 + t12;
  const double t14 = 0.0010000000474974513 * t13;
  const double t15 = PF_DIV(t14, vUII);
  vDUII = t15;
  vUIII = 7.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_78(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0002789999998640269 * vT;
  const double t1 = 1.2400000095367432 + t0;
  vUI = t1;
  const double t3 = vY * 0.0016586000565439463;
  const double t4 = 0.0028438998851925135 + t3;
  const double t5 = vY * t4;
  const double t6 = -0.04080900177359581 + t5;
  const double t7 = vY * t6;
  const double t8 = 1.0546000003814697 + t7;
  vUII = t8;
  vUIII = 7.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_79(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 1.0;
  vUII = 2.0;
  const double t0 = 3.9760001527611166e-05 * vT;
  const double t1 = 0.6690000295639038 + t0;
  const double t2 = pf_amax1(1.0, t1);
  vUIII = t2;
  const double t3 = PF_DIV(3.9760001527611166e-05, vUIII);
  const double t4 = (vUIII != 1.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUIII;
  vDUIII = t5;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_79(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 1.0;
  vUII = 2.0;
  const double t0 = 3.9760001527611166e-05 * vT;
  const double t1 = 0.6690000295639038 + t0;
  const double t2 = pf_amax1(1.0, t1);
  vUIII = t2;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_80(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.0003349999897181988 * vT;
  const double t1 = 0.6299999952316284 + t0;
  const double t2 = pf_amax1(2.0, t1);
  vUI = t2;
  const double t3 = PF_DIV(0.0003349999897181988, vUI);
  const double t4 = (vUI != 2.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  vUII = 1.0;
  vUIII = 2.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_80(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.0003349999897181988 * vT;
  const double t1 = 0.6299999952316284 + t0;
  const double t2 = pf_amax1(2.0, t1);
  vUI = t2;
  vUII = 1.0;
  vUIII = 2.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_81(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.00023499999952036887 * vT;
  const double t1 = 0.41999998688697815 + t0;
  const double t2 = pf_amax1(1.0, t1);
  vUI = t2;
  const double t3 = PF_DIV(0.00023499999952036887, vUI);
  const double t4 = (vUI != 1.0) ? 1.0 : 0.0;
  const double t5 = (t4 != 0.0) ? t3 : vDUI;
  vDUI = t5;
  const double t6 = 0.0005000000237487257 * vT;
  const double t7 = -1.2000000476837158 + t6;
  const double t8 = (vT > 6125.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t10 = PF_DIV(0.0005000000237487257, vUI);
  const double t11 = (vT > 6125.0) ? 1.0 : 0.0;
  const double t12 = (t11 != 0.0) ? t10 : vDUI;
  vDUI = t12;
  const double t13 = 7.899999764049426e-05 * vT;
  const double t14 = 1.7200000286102295 + t13;
  const double t15 = pf_amax1(2.0, t14);
  vUII = t15;
  const double t16 = PF_DIV(7.899999764049426e-05, vUII);
  const double t17 = (vUII != 2.0) ? 1.0 : 0.0;
  const double t18 = (t17 != 0.0) ? t16 : vDUII;
  vDUII = t18;
  vUIII = 1.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_81(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.00023499999952036887 * vT;
  const double t1 = 0.41999998688697815 + t0;
  const double t2 = pf_amax1(1.0, t1);
  vUI = t2;
  const double t6 = 0.0005000000237487257 * vT;
  const double t7 = -1.2000000476837158 + t6;
  const double t8 = (vT > 6125.0) ? 1.0 : 0.0;
  const double t9 = (t8 != 0.0) ? t7 : vUI;
  vUI = t9;
  const double t13 = 7.899999764049426e-05 * vT;
  const double t14 = 1.7200000286102295 + t13;
  const double t15 = pf_amax1(2.0, t14);
  vUII = t15;
  vUIII = 1.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_82(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  const double t0 = 0.00028700000257231295 * vT;
  const double t1 = 2.7799999713897705 + t0;
  vUI = t1;
  const double t2 = PF_DIV(0.00028700000257231295, vUI);
  vDUI = t2;
  const double t3 = 0.00014099999680183828 * vT;
  const double t4 = 0.3700000047683716 + t3;
  const double t5 = pf_amax1(1.0, t4);
  vUII = t5;
  const double t6 = PF_DIV(0.00014099999680183828, vUII);
  const double t7 = (vUII != 1.0) ? 1.0 : 0.0;
  const double t8 = (t7 != 0.0) ? t6 : vDUII;
  vDUII = t8;
  vUIII = 2.5;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_82(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  const double t0 = 0.00028700000257231295 * vT;
  const double t1 = 2.7799999713897705 + t0;
  vUI = t1;
  const double t3 = 0.00014099999680183828 * vT;
  const double t4 = 0.3700000047683716 + t3;
  const double t5 = pf_amax1(1.0, t4);
  vUII = t5;
  vUIII = 2.5;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_83(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 5.0;
  vUII = 5.0;
  vUIII = 4.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_83(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 5.0;
  vUII = 5.0;
  vUIII = 4.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_84(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 4.0;
  vUII = 6.0;
  vUIII = 6.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_84(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 4.0;
  vUII = 6.0;
  vUIII = 6.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_85(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 1.0;
  vUII = 4.0;
  vUIII = 6.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_85(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 1.0;
  vUII = 4.0;
  vUIII = 6.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_86(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 2.0;
  vUII = 1.0;
  vUIII = 4.5;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_86(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 2.0;
  vUII = 1.0;
  vUIII = 4.5;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_87(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 1.0;
  vUII = 2.0;
  vUIII = 1.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_87(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 1.0;
  vUII = 2.0;
  vUIII = 1.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_88(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 6.0;
  vUII = 3.0;
  vUIII = 7.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_88(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 6.0;
  vUII = 3.0;
  vUIII = 7.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_89(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 8.0;
  vUII = 8.0;
  vUIII = 8.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_89(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 8.0;
  vUII = 8.0;
  vUIII = 8.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_90(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 50.0;
  vUII = 50.0;
  vUIII = 50.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_90(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 50.0;
  vUII = 50.0;
  vUIII = 50.0;
  return PfVal{{vUI, vUII, vUIII}};
}

__device__ __noinline__ PfOut pf_elem_91(double vT, double vX, double vY, double vDX) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0, vDUI = 0.0, vDUII = 0.0, vDUIII = 0.0;
  (void)vT; (void)vX; (void)vY; (void)vDX;
  vUI = 25.0;
  vUII = 25.0;
  vUIII = 25.0;
  return PfOut{{vUI, vUII, vUIII}, {vDUI, vDUII, vDUIII}};
}

__device__ __noinline__ PfVal pf_value_91(double vT, double vX, double vY) {
#pragma clang fp contract(off)
  double vUI = 0.0, vUII = 0.0, vUIII = 0.0;
  (void)vT; (void)vX; (void)vY;
  vUI = 25.0;
  vUII = 25.0;
  vUIII = 25.0;
  return PfVal{{vUI, vUII, vUIII}};
}

// The same without derivatives, vX = log(5040 / T) and vY = 1e-3 T given
__device__ __forceinline__ void partition_values(int elem, double vT, double vX, double vY, double u[3]) {
  PfVal r = {{0.0, 0.0, 0.0}};
  switch (elem) {
    case 0: r = pf_value_0(vT, vX, vY); break;
    case 1: r = pf_value_1(vT, vX, vY); break;
    case 2: r = pf_value_2(vT, vX, vY); break;
    case 3: r = pf_value_3(vT, vX, vY); break;
    case 4: r = pf_value_4(vT, vX, vY); break;
    case 5: r = pf_value_5(vT, vX, vY); break;
    case 6: r = pf_value_6(vT, vX, vY); break;
    case 7: r = pf_value_7(vT, vX, vY); break;
    case 8: r = pf_value_8(vT, vX, vY); break;
    case 9: r = pf_value_9(vT, vX, vY); break;
    case 10: r = pf_value_10(vT, vX, vY); break;
    case 11: r = pf_value_11(vT, vX, vY); break;
    case 12: r = pf_value_12(vT, vX, vY); break;
    case 13: r = pf_value_13(vT, vX, vY); break;
    case 14: r = pf_value_14(vT, vX, vY); break;
    case 15: r = pf_value_15(vT, vX, vY); break;
    case 16: r = pf_value_16(vT, vX, vY); break;
    case 17: r = pf_value_17(vT, vX, vY); break;
    case 18: r = pf_value_18(vT, vX, vY); break;
    case 19: r = pf_value_19(vT, vX, vY); break;
    case 20: r = pf_value_20(vT, vX, vY); break;
    case 21: r = pf_value_21(vT, vX, vY); break;
    case 22: r = pf_value_22(vT, vX, vY); break;
    case 23: r = pf_value_23(vT, vX, vY); break;
    case 24: r = pf_value_24(vT, vX, vY); break;
    case 25: r = pf_value_25(vT, vX, vY); break;
    case 26: r = pf_value_26(vT, vX, vY); break;
    case 27: r = pf_value_27(vT, vX, vY); break;
    case 28: r = pf_value_28(vT, vX, vY); break;
    case 29: r = pf_value_29(vT, vX, vY); break;
    case 30: r = pf_value_30(vT, vX, vY); break;
    case 31: r = pf_value_31(vT, vX, vY); break;
    case 32: r = pf_value_32(vT, vX, vY); break;
    case 33: r = pf_value_33(vT, vX, vY); break;
    case 34: r = pf_value_34(vT, vX, vY); break;
    case 35: r = pf_value_35(vT, vX, vY); break;
    case 36: r = pf_value_36(vT, vX, vY); break;
    case 37: r = pf_value_37(vT, vX, vY); break;
    case 38: r = pf_value_38(vT, vX, vY); break;
    case 39: r = pf_value_39(vT, vX, vY); break;
    case 40: r = pf_value_40(vT, vX, vY); break;
    case 41: r = pf_value_41(vT, vX, vY); break;
    case 42: r = pf_value_42(vT, vX, vY); break;
    case 43: r = pf_value_43(vT, vX, vY); break;
    case 44: r = pf_value_44(vT, vX, vY); break;
    case 45: r = pf_value_45(vT, vX, vY); break;
    case 46: r = pf_value_46(vT, vX, vY); break;
    case 47: r = pf_value_47(vT, vX, vY); break;
    case 48: r = pf_value_48(vT, vX, vY); break;
    case 49: r = pf_value_49(vT, vX, vY); break;
    case 50: r = pf_value_50(vT, vX, vY); break;
    case 51: r = pf_value_51(vT, vX, vY); break;
    case 52: r = pf_value_52(vT, vX, vY); break;
    case 53: r = pf_value_53(vT, vX, vY); break;
    case 54: r = pf_value_54(vT, vX, vY); break;
    case 55: r = pf_value_55(vT, vX, vY); break;
    case 56: r = pf_value_56(vT, vX, vY); break;
    case 57: r = pf_value_57(vT, vX, vY); break;
    case 58: r = pf_value_58(vT, vX, vY); break;
    case 59: r = pf_value_59(vT, vX, vY); break;
    case 60: r = pf_value_60(vT, vX, vY); break;
    case 61: r = pf_value_61(vT, vX, vY); break;
    case 62: r = pf_value_62(vT, vX, vY); break;
    case 63: r = pf_value_63(vT, vX, vY); break;
    case 64: r = pf_value_64(vT, vX, vY); break;
    case 65: r = pf_value_65(vT, vX, vY); break;
    case 66: r = pf_value_66(vT, vX, vY); break;
    case 67: r = pf_value_67(vT, vX, vY); break;
    case 68: r = pf_value_68(vT, vX, vY); break;
    case 69: r = pf_value_69(vT, vX, vY); break;
    case 70: r = pf_value_70(vT, vX, vY); break;
    case 71: r = pf_value_71(vT, vX, vY); break;
    case 72: r = pf_value_72(vT, vX, vY); break;
    case 73: r = pf_value_73(vT, vX, vY); break;
    case 74: r = pf_value_74(vT, vX, vY); break;
    case 75: r = pf_value_75(vT, vX, vY); break;
    case 76: r = pf_value_76(vT, vX, vY); break;
    case 77: r = pf_value_77(vT, vX, vY); break;
    case 78: r = pf_value_78(vT, vX, vY); break;
    case 79: r = pf_value_79(vT, vX, vY); break;
    case 80: r = pf_value_80(vT, vX, vY); break;
    case 81: r = pf_value_81(vT, vX, vY); break;
    case 82: r = pf_value_82(vT, vX, vY); break;
    case 83: r = pf_value_83(vT, vX, vY); break;
    case 84: r = pf_value_84(vT, vX, vY); break;
    case 85: r = pf_value_85(vT, vX, vY); break;
    case 86: r = pf_value_86(vT, vX, vY); break;
    case 87: r = pf_value_87(vT, vX, vY); break;
    case 88: r = pf_value_88(vT, vX, vY); break;
    case 89: r = pf_value_89(vT, vX, vY); break;
    case 90: r = pf_value_90(vT, vX, vY); break;
    case 91: r = pf_value_91(vT, vX, vY); break;
    default: break;
  }
  u[0] = r.u[0]; u[1] = r.u[1]; u[2] = r.u[2];
}

// U_I, U_II, U_III and their d ln U / dT at T for element elem (0-based)
__device__ __forceinline__ void partition_at(int elem, double vT, double vX, double vY, double vDX, double u[3],
                                             double du[3]) {
  PfOut r = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
  switch (elem) {
    case 0: r = pf_elem_0(vT, vX, vY, vDX); break;
    case 1: r = pf_elem_1(vT, vX, vY, vDX); break;
    case 2: r = pf_elem_2(vT, vX, vY, vDX); break;
    case 3: r = pf_elem_3(vT, vX, vY, vDX); break;
    case 4: r = pf_elem_4(vT, vX, vY, vDX); break;
    case 5: r = pf_elem_5(vT, vX, vY, vDX); break;
    case 6: r = pf_elem_6(vT, vX, vY, vDX); break;
    case 7: r = pf_elem_7(vT, vX, vY, vDX); break;
    case 8: r = pf_elem_8(vT, vX, vY, vDX); break;
    case 9: r = pf_elem_9(vT, vX, vY, vDX); break;
    case 10: r = pf_elem_10(vT, vX, vY, vDX); break;
    case 11: r = pf_elem_11(vT, vX, vY, vDX); break;
    case 12: r = pf_elem_12(vT, vX, vY, vDX); break;
    case 13: r = pf_elem_13(vT, vX, vY, vDX); break;
    case 14: r = pf_elem_14(vT, vX, vY, vDX); break;
    case 15: r = pf_elem_15(vT, vX, vY, vDX); break;
    case 16: r = pf_elem_16(vT, vX, vY, vDX); break;
    case 17: r = pf_elem_17(vT, vX, vY, vDX); break;
    case 18: r = pf_elem_18(vT, vX, vY, vDX); break;
    case 19: r = pf_elem_19(vT, vX, vY, vDX); break;
    case 20: r = pf_elem_20(vT, vX, vY, vDX); break;
    case 21: r = pf_elem_21(vT, vX, vY, vDX); break;
    case 22: r = pf_elem_22(vT, vX, vY, vDX); break;
    case 23: r = pf_elem_23(vT, vX, vY, vDX); break;
    case 24: r = pf_elem_24(vT, vX, vY, vDX); break;
    case 25: r = pf_elem_25(vT, vX, vY, vDX); break;
    case 26: r = pf_elem_26(vT, vX, vY, vDX); break;
    case 27: r = pf_elem_27(vT, vX, vY, vDX); break;
    case 28: r = pf_elem_28(vT, vX, vY, vDX); break;
    case 29: r = pf_elem_29(vT, vX, vY, vDX); break;
    case 30: r = pf_elem_30(vT, vX, vY, vDX); break;
    case 31: r = pf_elem_31(vT, vX, vY, vDX); break;
    case 32: r = pf_elem_32(vT, vX, vY, vDX); break;
    case 33: r = pf_elem_33(vT, vX, vY, vDX); break;
    case 34: r = pf_elem_34(vT, vX, vY, vDX); break;
    case 35: r = pf_elem_35(vT, vX, vY, vDX); break;
    case 36: r = pf_elem_36(vT, vX, vY, vDX); break;
    case 37: r = pf_elem_37(vT, vX, vY, vDX); break;
    case 38: r = pf_elem_38(vT, vX, vY, vDX); break;
    case 39: r = pf_elem_39(vT, vX, vY, vDX); break;
    case 40: r = pf_elem_40(vT, vX, vY, vDX); break;
    case 41: r = pf_elem_41(vT, vX, vY, vDX); break;
    case 42: r = pf_elem_42(vT, vX, vY, vDX); break;
    case 43: r = pf_elem_43(vT, vX, vY, vDX); break;
    case 44: r = pf_elem_44(vT, vX, vY, vDX); break;
    case 45: r = pf_elem_45(vT, vX, vY, vDX); break;
    case 46: r = pf_elem_46(vT, vX, vY, vDX); break;
    case 47: r = pf_elem_47(vT, vX, vY, vDX); break;
    case 48: r = pf_elem_48(vT, vX, vY, vDX); break;
    case 49: r = pf_elem_49(vT, vX, vY, vDX); break;
    case 50: r = pf_elem_50(vT, vX, vY, vDX); break;
    case 51: r = pf_elem_51(vT, vX, vY, vDX); break;
    case 52: r = pf_elem_52(vT, vX, vY, vDX); break;
    case 53: r = pf_elem_53(vT, vX, vY, vDX); break;
    case 54: r = pf_elem_54(vT, vX, vY, vDX); break;
    case 55: r = pf_elem_55(vT, vX, vY, vDX); break;
    case 56: r = pf_elem_56(vT, vX, vY, vDX); break;
    case 57: r = pf_elem_57(vT, vX, vY, vDX); break;
    case 58: r = pf_elem_58(vT, vX, vY, vDX); break;
    case 59: r = pf_elem_59(vT, vX, vY, vDX); break;
    case 60: r = pf_elem_60(vT, vX, vY, vDX); break;
    case 61: r = pf_elem_61(vT, vX, vY, vDX); break;
    case 62: r = pf_elem_62(vT, vX, vY, vDX); break;
    case 63: r = pf_elem_63(vT, vX, vY, vDX); break;
    case 64: r = pf_elem_64(vT, vX, vY, vDX); break;
    case 65: r = pf_elem_65(vT, vX, vY, vDX); break;
    case 66: r = pf_elem_66(vT, vX, vY, vDX); break;
    case 67: r = pf_elem_67(vT, vX, vY, vDX); break;
    case 68: r = pf_elem_68(vT, vX, vY, vDX); break;
    case 69: r = pf_elem_69(vT, vX, vY, vDX); break;
    case 70: r = pf_elem_70(vT, vX, vY, vDX); break;
    case 71: r = pf_elem_71(vT, vX, vY, vDX); break;
    case 72: r = pf_elem_72(vT, vX, vY, vDX); break;
    case 73: r = pf_elem_73(vT, vX, vY, vDX); break;
    case 74: r = pf_elem_74(vT, vX, vY, vDX); break;
    case 75: r = pf_elem_75(vT, vX, vY, vDX); break;
    case 76: r = pf_elem_76(vT, vX, vY, vDX); break;
    case 77: r = pf_elem_77(vT, vX, vY, vDX); break;
    case 78: r = pf_elem_78(vT, vX, vY, vDX); break;
    case 79: r = pf_elem_79(vT, vX, vY, vDX); break;
    case 80: r = pf_elem_80(vT, vX, vY, vDX); break;
    case 81: r = pf_elem_81(vT, vX, vY, vDX); break;
    case 82: r = pf_elem_82(vT, vX, vY, vDX); break;
    case 83: r = pf_elem_83(vT, vX, vY, vDX); break;
    case 84: r = pf_elem_84(vT, vX, vY, vDX); break;
    case 85: r = pf_elem_85(vT, vX, vY, vDX); break;
    case 86: r = pf_elem_86(vT, vX, vY, vDX); break;
    case 87: r = pf_elem_87(vT, vX, vY, vDX); break;
    case 88: r = pf_elem_88(vT, vX, vY, vDX); break;
    case 89: r = pf_elem_89(vT, vX, vY, vDX); break;
    case 90: r = pf_elem_90(vT, vX, vY, vDX); break;
    case 91: r = pf_elem_91(vT, vX, vY, vDX); break;
    default: break;
  }
  u[0] = r.u[0]; u[1] = r.u[1]; u[2] = r.u[2];
  du[0] = r.du[0]; du[1] = r.du[1]; du[2] = r.du[2];
}

__device__ __forceinline__ void partition_gen(int elem, double T, double u[3], double du[3]) {
  partition_at(elem, T, log(5040.0 / T), 1.0e-3 * T, -1.0 / T, u, du);
}

}  // namespace fz
