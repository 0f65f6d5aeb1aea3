// Generated by gen_kernel_fits.py -- do not edit.
#pragma once
// Gaussian-erf reduced functions on t = q^2 in [0, 2.25]
static constexpr float kErfFitTMax = 2.25f;
// kErfPhi0: degree 7 in t, max rel. error of FP32 Horner 1.4e-07
static constexpr float kErfPhi0[8] = {2.659615278e-01f, -7.978845388e-02f, 1.424790546e-02f, -1.846842235e-03f, 1.886999526e-04f, -1.580060962e-05f, 1.056344786e-06f, -4.396050457e-08f};

// kErfPhi1: degree 7 in t, max rel. error of FP32 Horner 1.7e-07
static constexpr float kErfPhi1[8] = {5.319230258e-02f, -1.899725012e-02f, 3.693899838e-03f, -5.036801449e-04f, 5.321832941e-05f, -4.561751666e-06f, 3.098160448e-07f, -1.300545982e-08f};

// Gaussian-erf S = q erfc(q/sqrt2) e^{q^2/2} on w = 1/q in [1/7, 2/3]
// kErfcS: degree 8 in w, max rel. error of FP32 Horner 2.1e-07
static constexpr float kErfcS[9] = {7.978269458e-01f, 7.413595449e-04f, -7.900641561e-01f, -2.302378118e-01f, 4.490839005e+00f, -9.848020554e+00f, 1.109298992e+01f, -6.728021622e+00f, 1.744396210e+00f};

// Gaussian-erf phi2 on t = q^2 in [0, 4] (adjoint)
static constexpr float kErfPhi2TMax = 4.0f;
// kErfPhi2: degree 9 in t, max rel. error of FP32 Horner 6.7e-07
static constexpr float kErfPhi2[10] = {1.139835119e-01f, -4.432692006e-02f, 9.066865779e-03f, -1.278648037e-03f, 1.385016803e-04f, -1.220467857e-05f, 9.014397619e-07f, -5.541026837e-08f, 2.586244996e-09f, -6.734517805e-11f};

// Gaussian reduced functions on u = q^3 in [0, 1]
static constexpr float kGauFitUMax = 1.0f;
// kGauPhi0: degree 7 in u, max rel. error of FP32 Horner 1.2e-07
static constexpr float kGauPhi0[8] = {1.000000000e+00f, -5.000000000e-01f, 1.666664928e-01f, -4.166531935e-02f, 8.328105323e-03f, -1.377711771e-03f, 1.849033724e-04f, -1.591999171e-05f};

// kGauPsi: degree 7 in u, max rel. error of FP32 Horner 1.6e-07
static constexpr float kGauPsi[8] = {5.000000000e-01f, -3.333333135e-01f, 1.249998361e-01f, -3.333208337e-02f, 6.939634215e-03f, -1.180276740e-03f, 1.613655040e-04f, -1.403532951e-05f};

// kGauChi: degree 8 in u, max error / max|chi| of FP32 Horner 2.7e-07
static constexpr float kGauChi[9] = {-1.500000000e+00f, 4.000000000e+00f, -2.624999523e+00f, 9.999954700e-01f, -2.708097100e-01f, 5.707337335e-02f, -9.774587117e-03f, 1.329398714e-03f, -1.125588024e-04f};

// FP64, Gaussian-erf: phi1 on t = q^2 in [0, 4], S on w = 1/q in [0.1, 0.5]
static constexpr double kErf64TMax = 4.0, kErf64TMid = 2.0, kErf64WMid = 0.35;
// kErf64Phi1: degree 14 in t - 2, max weighted error 1.9e-16
static constexpr double kErf64Phi1[15] = {2.66676419900561158e-02, -8.87410862528015959e-03, 1.64973408154764161e-03, -2.18115400231975066e-04, 2.25561925434028513e-05, -1.92171064162084224e-06, 1.39417941685833057e-07, -8.81437819454510964e-09, 4.94022751046622183e-10, -2.48736000040125539e-11, 1.13698922364128652e-12, -4.75885969840971219e-14, 1.83810766785130326e-15, -6.68739341771007786e-17, 2.18784717775078739e-18};

// kErf64S: degree 13 in w - 0.35, max weighted error 2.1e-17
static constexpr double kErf64S[14] = {7.23555060735922462e-01, -3.33667518908424665e-01, -1.08733986486557160e-01, 4.84637334808815490e-01, -6.21153760397772481e-01, 3.29746491323714308e-01, 5.01667673483069509e-01, -1.75106977853493495e+00, 2.85783844743687432e+00, -2.65236212829008755e+00, -6.41369989015191155e-01, 8.88867818303855373e+00, -2.04861033696686299e+01, 2.10918241045758066e+01};

// e^x on |x| <= ln(2)/2, and ln 2 = hi + lo (hi of 32 bits: k hi is exact)
static constexpr double kLn2Hi = 6.93147180369123816e-01, kLn2Lo = 1.90821492927058770e-10;
// kExp64: degree 11 in x, max weighted error 2.4e-17
static constexpr double kExp64[12] = {1.00000000000000000e+00, 1.00000000000000000e+00, 5.00000000000001776e-01, 1.66666666666661467e-01, 4.16666666664930463e-02, 8.33333333356924000e-03, 1.38888889511617889e-03, 1.98412694136199634e-04, 2.48014865772065578e-05, 2.75576384411715744e-06, 2.76322758532418786e-07, 2.49894818233006896e-08};

